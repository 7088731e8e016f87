// Persistent unpack engine: one long-running gfx950 kernel per GPU that turns slots published in mapped host
// memory into scatter-gather copies and reports completion into mapped host memory -- no launch per request.
//
// Roles inside the one kernel launch
//   workgroup 0, wavefront 0  "leader": polls the submission ring over PCIe (sixteen entries per round trip),
//                             cuts each submission into tickets of 8 to 16 consecutive descriptors (by backlog;
//                             up to 64 where the payload says the fragments are short; or of the fixed
//                             `descs_per_ticket`) and writes them into a device-memory ticket ring: several
//                             waiting submissions at once where it can.  It never copies payload.
//   every other workgroup     "worker": one fetcher wavefront claims the next ticket number with one atomic,
//                             polls that ticket's slot until its stamps match, reads the ticket's descriptors
//                             (one per lane) and leaves in LDS, per fragment, a record of what the copy needs
//                             to know about it (which destination lines it shares with its neighbours, in
//                             the ticket and, when the engine is busy, in the tickets before and after);
//                             the copy wavefronts copy the fragments from those records,
//                             and the last of them to finish counts the ticket done.  Whoever counts the last
//                             ticket of a submission writes the completion word that the host poller reads.
//
// No cache maintenance.  Nothing here uses an acquire or release fence: on this GPU those become L2 write-back
// and invalidate instructions, and thousands of pollers issuing them stall everybody.  Instead every access
// to shared state carries its own coherence: control words and tickets are read and written with system-scope
// (sc0 sc1) accesses that bypass the per-XCD L2, payload is loaded and stored the same way, and ordering comes
// from s_waitcnt: a wavefront drains its store counter before the workgroup counts a ticket done.
// Records that are written by one side and polled by the other (host submissions, tickets) are 64 bytes in four
// 16-byte sectors, each ending in a stamp derived from the record's sequence number; a reader accepts a record
// only when all four stamps match, so a record is valid even if its sectors arrive as separate transactions,
// and the writer never has to order "payload, then flag".
//
// Liveness: no workgroup ever waits for another worker.  Workers wait only for the leader (their ticket) and
// watch the stop word while they do; the leader waits for nothing (a full ticket ring or job table just defers
// a submission to a later poll, and the leader asks for what is done before that one).  The host stop word, or the optional spin limit, ends the leader; the leader
// drains its stores, then sets the stop words; a worker that sees one looks at its ticket a last time and leaves.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "engine_rules.h"
#include "hip_common.h"
#include "tcpx_unpack_hip.h"
#include "unpack_device.h"

namespace tcpxu {
namespace {

constexpr uint32_t kMaxDescsPerSubmission = 1u << 20;
constexpr uint32_t kSmallestAdaptiveTicket = 8;  // the least ticket_size_for_submission returns
// The most descriptors one submission may carry: all its tickets must fit the ticket ring at once, or the leader
// could never hand it out (it defers a submission until the ring has room for all of its tickets).
__host__ __device__ constexpr uint32_t max_descs_for(uint32_t fixed_per_ticket) {
  const uint64_t smallest = fixed_per_ticket != 0 ? fixed_per_ticket : kSmallestAdaptiveTicket;
  const uint64_t fit = smallest * kTicketRing;
  return fit < kMaxDescsPerSubmission ? static_cast<uint32_t>(fit) : kMaxDescsPerSubmission;
}
constexpr uint32_t kStopReplicas = 64;
constexpr uint32_t kPollEntries = 16;  // submission entries fetched per load instruction of a leader poll (16 B per lane)
// A poll that finds all sixteen entries there and turns them into tickets at a stroke is followed by a deep poll:
// four loads in flight together, 64 entries for the one PCIe round trip (about 1.5 us) that sixteen cost -- which
// is what capped a storm of one-ticket requests near 9 M/s.
constexpr uint32_t kDeepGroups = 3;    // groups of kPollEntries beyond the first in a deep poll
constexpr uint32_t kStormBacklog = 128;  // entries published beyond a poll's 64 from which the leader takes them in a rolling loop
constexpr uint32_t kStormMost = 1u << 24;  // entries after which that loop returns all the same (see leader_storm)
// Lanes of the auxiliary load, among those that read nothing of an entry's own (see leader_loop).
constexpr uint32_t kAuxHostStop = 2, kAuxJobsCompleted = 6, kAuxProbe = 10;
constexpr uint32_t kNeverIdleOut = 0xFFFFFFFFu;
constexpr uint32_t kDefaultIdlePolls = 400;  // empty polls (of 1.75 us) before the kernel leaves by itself
constexpr int kTcpxuInProgress = TCPXU_IN_PROGRESS;

// 64-byte record: four 16-byte sectors of three payload words and one stamp word.
struct alignas(64) Record {
  uint32_t w[16];
};
constexpr int kPayloadWords = 12;
__host__ __device__ constexpr int payload_slot(int i) { return (i / 3) * 4 + (i % 3); }
// Submission payload: 0-1 bounce, 2-3 dst, 4-5 descs, 6-7 done_flag, 8-9 done_value, 10 n_descs, 11 payload bytes
//                     (0 = not given).
// Ticket payload:     0-1 bounce, 2-3 dst, 4-5 descs, 6-7 done_flag, 8-9 done_value,
//                     10 n | job << 8 | before << 29 | after << 30 | only << 31, 11 target.
// `only`: the submission's only ticket (the job slot index is below 2^16); `before` / `after`: the submission has
// descriptors before this ticket's first / after its last (in the same array: the fetcher looks at the nearest one
// to decide whether the destination line at that end of the ticket is shared with the neighbouring ticket).
constexpr uint32_t kOnlyTicket = 1u << 31;
constexpr uint32_t kMoreAfter = 1u << 30, kMoreBefore = 1u << 29;
// Descriptors that travel with the submission.  A small request's descriptors lie in memory that the GPU reaches over
// PCIe (1.7 us from the ticket's record to the last of them, 0.8 if the caller has put a copy into the GPU's memory, which
// costs the caller a microsecond of waiting for its write-combining buffers).  The host has them at hand when it submits:
// where it can see that they are host memory it copies them beside the ring's entry, the leader fetches those of the
// next few entries in the round trip that fetches the entries, and writes them beside the ticket, where the fetcher that
// polls the ticket reads them in the same round trip as the record: 0.5 us.  (A lone request of 16 whole pages, publish ->
// done: 7.7 us -> 6.5 with the looks below.)  Each is one 16-byte sector of three words and the stamp of its entry or
// ticket, like the records' own: source offset, length, the destination offset's low word (a list with a destination
// offset of 4 GiB or more is not carried).  Sixteen, a ticket of which is a quarter of a look's lanes; only the first four
// of a call, and only while the leader keeps up, because only the first four entries of a look bring theirs and the copy
// costs the host 50 ns each (2048 requests in one call: 1 us in 67).
constexpr uint32_t kCarriedEntry = 1u << 31;   // in a submission's payload word 10, beside the count
// There too, of a submission of short fragments: how many more the same call hands over.  The leader looks at the ring
// faster than the host writes it, so the first submissions of a burst would be cut up as if each came alone (eleven
// requests of 2000 short fragments in one call: 28.4 -> 26.2 us).  Whole pages are not sized so: there
// small tickets reach all the workgroups sooner (32 requests of 2 MiB by what has been seen 35.1 us, and 36.5 with every one sized for all).
// And whether it is of a burst that burst_of_pages or burst_of_short_fragments names.  The host works that out, since every
// instruction that the leader spends on an entry is waited for by all that follow it.
constexpr uint32_t kBurstEntry = 1u << 30;
constexpr uint32_t kFollowShift = 21, kMostFollow = 0x1FF;
constexpr uint32_t kCountMask = (1u << kFollowShift) - 1u;  // 1 .. 2^20 descriptors
__device__ __forceinline__ uint32_t following(uint32_t count_word) { return (count_word >> kFollowShift) & kMostFollow; }
constexpr uint32_t kCarriedTicket = 1u << 28;  // in a ticket's
constexpr uint32_t kCarriedEntries = 4;        // entries of a poll whose descriptors it fetches as well: 64 lanes' worth
constexpr uint32_t kCarryBehind = 16;          // entries the leader is behind from which the host carries no more
// The least submission ring.  A look or poll brings kPollEntries entries, no two of which may share a place; and the host does not
// read the leader's position while, by the one it knows, the leader is kCarryBehind entries behind at most: a ring shorter than
// that could be full by the known position and not by the real one, and never be found otherwise.
constexpr uint32_t kSmallestRing = 16;
static_assert(kPollEntries <= kSmallestRing && kCarryBehind <= kSmallestRing, "what reads or writes the ring without asking");
// Looks at a ticket that is not there yet after which its fetcher asks for a carried list as well.  Small requests on an
// idle engine find fetchers that have waited long, and those are the ones whose descriptors are waited for; under load a
// ticket is there at one of the first looks, and 256 bytes more with each of those cost streams of large requests, which
// carry none: 1 MiB requests whose buffers stay in the caches 3.25 TB/s with every look asking, 3.37 after 1, 4 or 16 (3.38
// before lists travelled), the headline workload 71.8 and 72.0 %.  A list that was not asked for is read where it lies.
constexpr uint32_t kAskAfter = 4;
struct alignas(64) CarriedList {
  uint32_t w[kCarriedDescs][4];
};
// Whether a submission's tickets share destination lines across their ends.  It saves two partial writes of a line
// per ticket boundary and costs every ticket's pick-up two more descriptors to read and look at: worth it when the
// engine is busy (8 MiB workload +0.3 points of the roofline, fragments of 1.8 KiB +0.4), not for a request that is
// alone (4 MiB: 0.3 us more), and pointless where whole pages land on line boundaries anyway (1 MiB requests of
// whole pages: 0.90 -> 0.84 of the roofline with it).  Decided by the leader for the whole submission, so that the
// two tickets at a boundary always agree.
__host__ __device__ __forceinline__ bool shares_across_tickets(uint32_t in_flight, uint32_t n, uint32_t bytes,
                                                               uint32_t dst_lo) {
  const bool whole_pages_on_lines = bytes == n * TCPXU_PAGE_SIZE && (dst_lo & 127u) == 0;
  return in_flight >= kManyInFlight && !whole_pages_on_lines;
}

struct HostCtl {  // mapped host memory
  alignas(64) uint64_t tail;       // host -> GPU: submissions published so far
  alignas(64) uint64_t stop;       // host -> GPU: drain and exit
  alignas(64) uint64_t head;       // GPU -> host: submissions the leader has consumed
  alignas(64) uint64_t completed;  // GPU -> host: submissions fully unpacked (told with a look that finds nothing, if it has changed, and at exit)
  alignas(64) uint64_t exited;     // GPU -> host: 0 running, 1 stopped on request, 2 left after being idle
  alignas(64) uint64_t exiting;    // GPU -> host: the leader is about to leave for idleness (see leader_loop)
  // GPU -> host, written by the leader when it leaves: its polls of the ring, the entries they consumed and the
  // polls that fetched 64 entries instead of 16, since the engine was created.
  alignas(64) uint64_t leader_polls;
  uint64_t leader_entries;
  uint64_t leader_deep_polls;
  alignas(64) Record ring[1];      // ring_entries follow, then as many CarriedLists
};

struct alignas(256) StopWord {
  uint32_t value;
};

// The three words that every workgroup counts in, and one of which every look of the leader reads, lie 4 KiB apart: an atomic
// takes its memory channel 12 ns, and in one line they waited for each other and the looks for them.  (64 / 4096 bytes apart, us
// a call with other buffers from pass to pass: a request of 64 KiB 8.53 / 8.33, 256 of them 21.9 / 21.3, 64 MiB of ragged
// fragments 36.6 / 35.9, of wire fragments 32.7 / 32.3; a stream of 64 KiB requests, 256 in flight, 2.47 / 2.56 TB/s r+w; 256
// bytes apart measures the same but for that stream, 2.49.)
constexpr size_t kCountersApart = 4096;
struct alignas(256) Counter {
  uint64_t value;
  uint8_t apart[kCountersApart - sizeof(uint64_t)];
};
static_assert(sizeof(Counter) == kCountersApart, "no further apart than that");
struct DevState {  // device memory
  Counter ticket_head;     // next ticket number to claim
  Counter tickets_done;    // tickets whose payload is written
  Counter jobs_completed;  // submissions completed since creation
  alignas(64) uint64_t sub_head;        // leader-private: next submission index
  uint64_t tickets_out;                 // leader-private: tickets written so far
  uint64_t leader_polls, leader_entries, leader_deep_polls;  // leader-private: running totals (see HostCtl)
  alignas(64) uint32_t exited_wgs;      // reset at every start, as are the stop words
  uint32_t exit_reason;
  alignas(64) uint32_t leader_place;    // likewise: the leader's compute unit (see kEnoughElsewhere)
  uint32_t workers_elsewhere;           // worker workgroups that have started on other ones
  alignas(256) StopWord stop[kStopReplicas];
  alignas(64) Record tickets[kTicketRing];
  CarriedList carried[kTicketRing];  // of the tickets that say so
  // uint32_t jobs_done[ring_entries], then uint32_t job_target[ring_entries] follow: per job slot, the tickets counted and the
  // tickets ever issued of the submissions of several tickets that it has had.  (A submission's only ticket completes it
  // and is not counted there.)
};

// ---- scoped memory operations -------------------------------------------------------------------------------------
#define SYS __HIP_MEMORY_SCOPE_SYSTEM

template <typename T>
__device__ __forceinline__ T sys_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, SYS);
}
template <typename T>
__device__ __forceinline__ void sys_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, SYS);
}
// The same for memory that is known to be global (device memory, mapped host memory), said outright: where the
// compiler cannot see that -- a pointer that arrived as a function's argument -- it would emit a flat_ store, which
// the hardware is free to complete out of turn among a wavefront's memory instructions.
template <typename T>
__device__ __forceinline__ void sys_store_global(T* p, T v) {
  __hip_atomic_store((TCPXU_GLOBAL T*)p, v, __ATOMIC_RELAXED, SYS);  // (only a C-style cast changes the address space)
}
__device__ __forceinline__ void drain_memory_ops() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint32_t bcast(uint32_t v, uint32_t src_lane) {
  return __shfl(v, static_cast<int>(src_lane), kWaveLanes);
}
// ---- looks at the ring ----------------------------------------------------------------------------------------------
// A look brings sixteen entries, the descriptors that travel with the first four, and what is known of the entries' job
// slots, straight into LDS.  kLooks of them are under way at a time, so that an entry waits half the round trip to the
// host's memory (1.25 us, whatever it brings) less for the look that sees it, and going through one look hides behind the next;
// in LDS because a look that is still under way when the leader leaves this way of polling would otherwise land in registers that
// have found another use.
// What bounds a lone request here is how soon a look shows it and how soon it is a ticket then, and both are instructions of a
// single wavefront: a pass of the leader's whole loop takes 0.95 us, and while every look cost one, looks came round no sooner
// than that, however many were under way.  Hence a loop of their own that does the least: a look that shows nothing costs it
// 0.25 us, entries of one ticket each, wherever their descriptors lie, and entries of several, if few wait, are written there and
// then, and anything else leaves it.  Nor does a look read what the workgroups count in, beyond the count of completed
// submissions: their counting waits for it (see nothing_under_way).  (Us, before / now, buffers in turn: a request of 64 KiB of
// pages 8.30 / 7.70, through the plugin 7.35 / 6.88, 2048 of them through the plugin, 16 posted at a time, 1030 / 930; sixteen
// requests of 4 MiB 32.4 / 30.9; a hundred of 200 KB through the plugin, 4 posted at a time, 227 / 209.  A request alone at random
// times, publish -> done as the host sees it, 1 / 16 / 32 / 256 / 1024 pages: 5.45 / 6.5 / 7.5 / 7.65 / 8.85 before, 4.95 / 6.1 / 7.0 /
// 7.35 / 8.6 now.)
// Four under way, one each 0.38 us, are no faster for one request (6.20 and 6.25 over those sizes), and the 2048 take 990, since
// the host writes entries whose lines are being read.
// (A look asked for before an earlier one was gone through shows the job slots' counters as they were then.  That is safe:
// a ring has sixteen entries or more, so none of a look's entries shares its slot with another of them, and what was
// issued for the slot's last tenant was written before the look was asked for.)
constexpr uint32_t kLooks = 2;  // (a power of two: places are counted modulo it)
struct alignas(16) Look {
  uint32_t sect[kWaveLanes][4];     // lane 4k+j: sector j of entry base+k
  uint32_t carried[kWaveLanes][4];  // lane 16k+j: descriptor j of entry base+k
  uint32_t aux[kWaveLanes];         // see leader_loop
};
constexpr uint32_t kAskedBits = 16, kAskedMask = (1u << kAskedBits) - 1u;
static_assert(kLooks * kAskedBits <= 64, "leader_loop keeps them in one register");
static_assert(kCarriedEntries * kCarriedDescs == kWaveLanes, "a lane to a descriptor");
constexpr int kLookSleep = 2;  // in 64 clocks; 0 to 4 measured alike
constexpr uint32_t kLookLoads = 3;  // vector memory instructions of a look
// Entries in a look up to which those of several tickets are handed out one after the other where they are looked at.  From
// kLeaderBehindShallow on the leader counts as behind, and that is for its ordinary way.  (With 1 / 2 / 3 / 5 here: two ragged requests
// of 1 and 0.7 MB in one call 12.3 / 11.7 / 11.7 / 11.6 us, 12.1 before looks had a loop; a hundred of 200 KB through the plugin,
// 4 posted at a time, 209 / 207 / 205 / 205; six of 280 KB 12.0 / 12.2 / 12.2 / 12.4.)
constexpr uint32_t kFewReady = kLeaderBehindShallow - 1;
constexpr uint32_t kManyAtOnce = 3, kManySmall = 6;  // see where they are used
#define TCPXU_LDS __attribute__((address_space(3)))
typedef TCPXU_LDS Look LdsLook;
typedef TCPXU_LDS u32x4 lds_u32x4;
__device__ __forceinline__ uint32_t lds_address(const TCPXU_LDS void* p) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(reinterpret_cast<uintptr_t>(p))));
}
// The loads of a look (one address each per lane).  Instructions, because the compiler would wait for everything under way
// before the next read of LDS; m0 holds where in LDS lane 0's share goes.
__device__ __forceinline__ void ask_for_look(LdsLook* look, const void* aux, const uint8_t* carried, const uint8_t* sect) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 1\n\tglobal_load_lds_dword %3, off sc0 sc1\n\t"
      "s_mov_b32 m0, %1\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %4, off sc0 sc1\n\t"
      "s_mov_b32 m0, %2\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %5, off sc0 sc1"
      :
      : "s"(lds_address(look->aux)), "s"(lds_address(look->carried)), "s"(lds_address(look->sect)),
        "v"(reinterpret_cast<uint64_t>(aux)), "v"(reinterpret_cast<uint64_t>(carried)), "v"(reinterpret_cast<uint64_t>(sect))
      : "memory");
}

// ---- leader -------------------------------------------------------------------------------------------------------
// Runs on wavefront 0 of workgroup 0.  All control flow is wave-uniform.
__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t src_lane) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(src_lane)));
}

// Stamps (optional, tcpxuEngineEnableStamps): four 64-bit readings of the GPU's constant-rate clock per job slot, in
// device memory that the host has filled with ones -- [0] the leader saw the submission, [1] the first of its
// tickets was fetched by a workgroup, [2] the first workgroup had its descriptors staged (both kept as minima),
// [3] the workgroup that completed the submission had its last store acknowledged.
constexpr uint32_t kStampsPerJob = 4;
__device__ __forceinline__ uint64_t clock_now() { return wall_clock64(); }

// What the four lanes of an entry know about it, for the sixteen entries of one group at once.
struct EntryView {
  uint32_t n, bytes, per_ticket, target_prev, in_flight, slot;
  bool sane, slot_free;
};

// How many of a group's entries, from the first, can become tickets now, one each; `room` is what the ticket ring still
// takes.
__device__ __forceinline__ uint32_t single_tickets_run(const EntryView& v, uint32_t room) {
  const uint64_t not_now = ~__ballot(v.sane);
  const uint32_t run = not_now == 0 ? kPollEntries : static_cast<uint32_t>(__builtin_ctzll(not_now)) >> 2;
  return std::min(run, room);
}

// Every entry of a group fits one ticket (a storm of small requests): the leading run of them becomes tickets in
// one store instruction.  Returns the length of the run.
__device__ __forceinline__ uint32_t write_single_tickets_of_group(DevState* st, uint64_t* stamps, uint64_t& tickets_out,
                                                                  uint32_t lane, const EntryView& v, const u32x4& sc,
                                                                  uint32_t room) {
  const uint32_t k_of_lane = lane >> 2;
  const uint32_t run = single_tickets_run(v, room);
  if (run != 0) {
    if (k_of_lane < run) {
      const uint64_t t = tickets_out + k_of_lane;
      const uint32_t stamp = static_cast<uint32_t>(t + 1);
      u32x4 out{sc.x, sc.y, sc.z, stamp};
      if ((lane & 3u) == 3) {
        out.y = v.n | (v.slot << 8) | kOnlyTicket;
        if (stamps) sys_store_global(&stamps[kStampsPerJob * v.slot], clock_now());
      }
      store_vec_sys(reinterpret_cast<uint8_t*>(&st->tickets[t & (kTicketRing - 1)]) + 16 * (lane & 3u), out);
    }
    tickets_out += run;
  }
  return run;
}

// Where lanes that took different ways meet again, said as a statement of its own: where they meet at the end of a loop,
// the compiler would take whatever else meets there -- the leader's positions -- for different from lane to lane.
__device__ __forceinline__ void lanes_together() { asm volatile(""); }

// Every lane takes the value that lane q of its own group of four holds: one move, no trip through the LDS.
template <int q>
__device__ __forceinline__ uint32_t quad_value(uint32_t v) {
  static_assert(q >= 0 && q < 4, "a lane of the quad");
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), q * 0x55, 0xF, 0xF, false));
}

// The value `lanes` lanes below in the same row of sixteen, 0 where there is none.
template <int lanes>
__device__ __forceinline__ uint32_t row_shift(uint32_t v) {
  static_assert(lanes > 0 && lanes < 16, "within a row");
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x110 + lanes, 0xF, 0xF, true));
}

__device__ __forceinline__ uint32_t same_in_all_lanes32(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}
__device__ __forceinline__ uint64_t same_in_all_lanes64(uint64_t v) {
  return (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)))) << 32) |
         static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}
template <typename T>
__device__ __forceinline__ T* same_in_all_lanes_ptr(T* p) {
  return reinterpret_cast<T*>(same_in_all_lanes64(reinterpret_cast<uint64_t>(p)));
}

// A storm: a deep poll turned all its 64 entries into tickets and the host has published kStormBacklog entries beyond
// them -- or a poll wrote several tickets for each of its sixteen entries, none of them large, and more of the kind
// may wait.  Takes entries from s on for as long as they are published and are one ticket each; returns where it
// got to, which is where it started if the first group was not for it.
//
// kGroups (five) groups of sixteen entries are in flight at a time, and the registers of a group that has gone through
// take the group 16 x kGroups entries on at once (every group's loads bring the stamp of the last entry of the group
// that would be asked for next: entries are published in order, so if that one is there the whole group is).  The
// leader's time per group is then a fifth of the round trip to the host's ring or what it takes to turn a group into
// tickets, whichever is longer -- not their sum as in a poll (1024 requests of 64 KiB in flight: 21 -> 44 M
// requests/s, where the copy itself becomes the bound).  Every group has registers of its own (moving one that is
// still in flight to another register would wait for it), hence one step unrolled per group, with every index into
// the groups' arrays a constant.  When the host's tail is reached nothing more is asked for and the groups in flight
// go through: the loop ends with nothing in flight.
//
// The compiler would wait for everything in flight at the top of such a loop.  So the loop's loads are written as
// instructions, which it does not track, and each step waits for its own group by count: the memory instructions of
// a wavefront complete in the order issued, and between a group's loads and its turn the other kGroups - 1 groups
// have had theirs, each with two stores (the tickets, how far it has got) and, while the loop feeds, two loads:
// 4 x (kGroups - 1) instructions at the least, so "at most that many outstanding" means that the group's own loads
// have landed.  (More are issued when stamps are on, and the head word once a round: counting too few only waits for
// a little more than is needed; fewer would let a group be read before it has landed, so this function must not
// spill registers to memory -- the build checks the compiler's resource report for 0 bytes of scratch.)  Once the
// loop has stopped feeding, a group waits for everything.  The group's registers pass through a statement after the
// wait so that nothing reads them before it.
//
// A function of its own, not inlined, and called from the top of the leader's loop where little is live: with this
// loop inside the leader's, what the compiler did with the registers around it made every poll that never sees a
// storm 0.2 us slower.  The running count of finished tickets is read whenever the first groups are asked for: too few
// counted as done only ends the storm early.  The leader, whose own count of them is of before the storm, asks again once
// so many are out by that count that the ring may be half full -- which the counts' low words tell, since no storm goes on for
// more than kStormMost entries.  (The loop's count handed back with the rest costs a lone request 0.04 us, 2.40 -> 2.44 from its
// descriptors staged to its last store, in copy wavefronts whose instructions are the same and lie elsewhere.)
struct StormEnd {
  uint64_t s, tickets_out;
  uint32_t entries;  // taken off the ring
};
__device__ __attribute__((noinline)) StormEnd leader_storm(HostCtl* ctl_in, DevState* st_in, uint64_t* stamps_in, uint32_t ring_mask_in,
                                                          uint32_t fixed_per_ticket_in, uint64_t s_in, uint64_t tickets_out_in) {
  // Arguments arrive in vector registers.  These are the same in every lane and go back to scalar registers.
  HostCtl* ctl = same_in_all_lanes_ptr(ctl_in);
  DevState* st = same_in_all_lanes_ptr(st_in);
  uint64_t* stamps = same_in_all_lanes_ptr(stamps_in);
  const uint32_t ring_mask = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(ring_mask_in)));
  const uint32_t fixed_per_ticket = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(fixed_per_ticket_in)));
  uint64_t s = same_in_all_lanes64(s_in);
  uint64_t tickets_out = same_in_all_lanes64(tickets_out_in);
  const uint32_t lane = threadIdx.x;
  const uint32_t k_of_lane = lane >> 2;
  uint32_t consumed = 0, entries = 0;
  // Groups in flight: the round trip to the host's ring, 1.55 us, over what a group costs to turn into tickets, 0.36 us,
  // and one more.  (1024 requests of 64 KiB in flight: 40.3 M/s with four, 44.6 with five -- where the copy itself is
  // the bound -- and 45.5 with six, which spills registers; 384 in flight: 29.4, 27.2, 26.4.)
  constexpr uint32_t kGroups = 5;
  // Every lane also reads the stamp of the last entry of the group that would be asked for next (the probe).  What of a
  // lane's address does not change from group to group is worked out once (and hidden from the compiler, which would work it
  // out again in every step).
  uint64_t entry_base = reinterpret_cast<uint64_t>(&ctl->ring[0]) + 16 * (lane & 3);
  asm volatile("" : "+v"(entry_base));
  const uint64_t probe_base = reinterpret_cast<uint64_t>(&ctl->ring[0].w[15]);
  static_assert(sizeof(Record) == 64, "the shifts below");
  auto fetch_group_untracked = [&](u32x4& sc, uint32_t& ax, uint64_t s_g) {
    const uint32_t at_s = static_cast<uint32_t>(s_g);  // (the mask keeps low bits only)
    const uint64_t entry = entry_base + (static_cast<uint64_t>((at_s + k_of_lane) & ring_mask) << 6);
    const uint64_t at = probe_base + (static_cast<uint64_t>((at_s + (kGroups + 1) * kPollEntries - 1) & ring_mask) << 6);
    asm volatile("global_load_dword %0, %1, off sc0 sc1" : "=v"(ax) : "v"(at) : "memory");
    asm volatile("global_load_dwordx4 %0, %1, off sc0 sc1" : "=v"(sc) : "v"(entry) : "memory");
  };
  // kGroups while the loop feeds (that many groups in flight); once it has caught up with the host, the groups still
  // in flight that have not gone through: kGroups - 1, ..., 1, and at 0 the storm is over.
  uint32_t feeding = kGroups;
  u32x4 sc[kGroups];
  uint32_t ax[kGroups], tickets_done;
  bool queue_deep = false;
  // The first groups, from s on, and the running count of finished tickets: one round trip, waited for whole.
  auto arm = [&]() {
    feeding = kGroups;
#pragma unroll
    for (uint32_t g = 0; g < kGroups; ++g) fetch_group_untracked(sc[g], ax[g], s + g * kPollEntries);
    asm volatile("global_load_dword %0, %1, off sc0 sc1" : "=v"(tickets_done) : "v"(reinterpret_cast<const uint32_t*>(&st->tickets_done.value)) : "memory");
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(tickets_done) : : "memory");
#pragma unroll
    for (uint32_t g = 0; g < kGroups; ++g) asm volatile("" : "+v"(sc[g]), "+v"(ax[g]) : : "memory");
    tickets_done = same_in_all_lanes32(tickets_done);
    // The first group's probe: the 16 x (kGroups + 1) entries from s on are published, so the queue at the leader is deep.
    queue_deep = lane_value(ax[0], 2) == static_cast<uint32_t>(s + (kGroups + 1) * kPollEntries);
  };
  // One group through; false when the storm is over: nothing more in flight, or the group was not there whole or not
  // all of one ticket each (then whatever is in flight is dropped, and the leader's next poll asks again).
  auto pass = [&](u32x4& sc, uint32_t& ax) {
    // (While the loop feeds, the kGroups - 1 steps before this one all fed: it stops feeding once and for all.  The
    // first groups have landed, whichever wait they get.)
    if (feeding == kGroups) asm volatile("s_waitcnt vmcnt(%0)" : : "n"((kGroups - 1) * 4) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    asm volatile("" : "+v"(sc), "+v"(ax) : : "memory");
    const uint64_t s_g = s + consumed;
    const uint64_t okm = __ballot(sc.w == static_cast<uint32_t>(s_g + k_of_lane + 1));
    uint32_t run = 0;
    if ((okm & 0xFull) == 0xFull) {
      const uint32_t left = ticket_room(static_cast<uint32_t>(tickets_out), tickets_done);
      // With hundreds of submissions waiting, one of at most 32 descriptors is one ticket (see
      // ticket_size_for_submission; a fixed ticket size says so itself) -- and when the loop was armed with the entry
      // 16 x (kGroups + 1) ahead published, so is one of as many descriptors as a ticket holds: every workgroup has
      // work anyway, and a ticket per entry is what lets the leader keep up (1024 requests of 33 whole pages in
      // flight: 5.8 -> 33 M requests/s).  No sizing here, and a group with a larger one ends the storm and goes the
      // ordinary way.
      EntryView more{};  // (write_single_tickets_of_group looks at nothing but what is set here)
      more.n = quad_value<3>(sc.y) & kCountMask;  // payload word 10 sits in .y of sector 3
      more.sane = ((okm >> (4 * k_of_lane)) & 0xFull) == 0xFull && more.n - 1u < kMaxDescsPerSubmission;
      more.slot = static_cast<uint32_t>(s_g + k_of_lane) & ring_mask;
      const uint32_t one_ticket = fixed_per_ticket != 0 ? fixed_per_ticket : queue_deep ? kMaxDescsPerTicket : kSmallSubmission;
      if (__ballot(more.sane && more.n > one_ticket) == 0) run = write_single_tickets_of_group(st, stamps, tickets_out, lane, more, sc, left);
    }
    consumed += run;
    if (run != 0 && lane == 0) sys_store_global(&st->sub_head, s_g + run);  // (one of the two stores counted above)
    if (run != kPollEntries) return false;
    if (feeding == kGroups) {
      const uint64_t next = s_g + kGroups * kPollEntries;
      if (lane_value(ax, 2) == static_cast<uint32_t>(next + kPollEntries)) fetch_group_untracked(sc, ax, next);
      else feeding = kGroups - 1;
    } else {
      --feeding;
    }
    feeding = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(feeding)));
    return feeding != 0;
  };
  auto round = [&]() {
#pragma unroll
    for (uint32_t g = 0; g < kGroups; ++g)
      if (!pass(sc[g], ax[g])) return false;
    return true;
  };
#pragma unroll 1
  for (;;) {
    arm();
#pragma unroll 1
    for (;;) {
      if (!round()) break;
      // a round of entries on: the host learns of it
      s += consumed;
      entries += consumed;
      consumed = 0;
      if (lane == 0) sys_store_global(&ctl->head, s);
    }
    // Whatever is still in flight is waited for, so that the registers it lands in are free.
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#pragma unroll
    for (uint32_t g = 0; g < kGroups; ++g) asm volatile("" : "+v"(sc[g]), "+v"(ax[g]) : : "memory");
    if (consumed != 0) {  // the round that the loop ended in
      s += consumed;
      entries += consumed;
      consumed = 0;
      if (lane == 0) sys_store_global(&ctl->head, s);
    }
    // Caught up with the host, every group in flight gone through whole (16 x kGroups entries at the least since the
    // loop was armed): the host publishes as requests complete, so more is on its way -- ask again from here instead of
    // leaving, waiting for the ordinary loop to find 64 entries and as many again beyond them, and coming back.
    // Anything else -- a group not there whole, entries of more than one ticket, no room in the ticket ring --
    // is for the ordinary loop.
    if (feeding != 0 || entries >= kStormMost) break;
  }
  return StormEnd{s, tickets_out, entries};
}

__device__ void leader_loop(HostCtl* ctl, DevState* st, uint32_t* jobs_done, uint32_t* job_target,
                            uint32_t ring_mask, uint32_t fixed_per_ticket, uint32_t spin_limit, uint64_t* stamps,
                            LdsLook* looks) {
  // The leader's positions are the same in every lane: said outright, so that they stay in scalar registers (in
  // vector registers the compiler waits for the leader's own stores at the top of every pass).
  auto same_in_all_lanes = [](uint64_t v) {
    return (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)))) << 32) |
           static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
  };
  uint64_t s = same_in_all_lanes(sys_load(&st->sub_head));
  uint64_t tickets_out = same_in_all_lanes(sys_load(&st->tickets_out));
  uint64_t mirrored = same_in_all_lanes(sys_load(&st->jobs_completed.value));  // completed submissions, as the host was last told
  // Read once: the grid's size comes from the dispatch packet, a scalar load with a wait behind it wherever it is asked.
  const uint32_t workers = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(gridDim.x - 1)));
  uint32_t idle = 0;
  // spin_limit counts polls that ask when the last is done, one in 1.75 us; looks are gone through every 0.75.
  const uint32_t idle_limit = spin_limit == kNeverIdleOut ? kNeverIdleOut : static_cast<uint32_t>(std::min<uint64_t>(7ull * spin_limit / 3, kNeverIdleOut - 1u));
  uint32_t reason = 0;
  uint32_t polls = 0, entries = 0, deep_polls = 0;  // of this launch; added to the running totals at the end
  uint32_t wide = 0;       // the last entry taken was one of several tickets, with none on its way that count for the size
  uint32_t direct = 0;     // the next poll brings its entries into registers (flags in scalar registers, like the positions)
  uint32_t deep = 0;       // and so many as 64 of them (a ring of fewer never has them)
  uint32_t under_way = 0;  // looks asked for and not gone through
  uint32_t look = 0;       // the next to ask for, modulo kLooks
  uint64_t asked_at = 0;   // the low bits of the first entry's number of each, the youngest's lowest
  // A word that workgroups count in is not one to look at all the time: reading it makes their counting wait (sixteen requests of
  // 4 MiB, looks every 0.75 us: 32.8 us with looks that read the finished tickets' count and the job slots', which share their
  // lines with those being counted in, 31.3 without; looks every 0.38 us 51 and 30.7).  So two facts are kept instead.
  // The low word of the tickets known to be done: all of them when nothing is under way, otherwise asked for as
  // ask_what_is_done says.
  uint32_t tickets_done = static_cast<uint32_t>(tickets_out);
  // Entries below this one have job slots known to be free: what is counted there is then what has been issued.
  uint64_t free_until = s + ring_mask + 1u;
  auto nothing_under_way = [&]() {  // every submission before entry s is completed (see known_done_after)
    tickets_done = static_cast<uint32_t>(tickets_out);
    free_until = s + ring_mask + 1u;
  };
  auto ask_done = [&]() { tickets_done = known_done_after(tickets_done, same_in_all_lanes32(static_cast<uint32_t>(sys_load(&st->tickets_done.value)))); };
  auto too_many_out = [&]() { return ask_what_is_done(static_cast<uint32_t>(tickets_out), tickets_done, false); };
  // The tickets of one submission of at least one descriptor, entry s_k, sixteen of them to a store instruction; false if they
  // cannot be written now.  `too_small`: see kLeaderBehind.
  auto write_tickets = [&](uint64_t s_k, u32x4 v, uint32_t count_word, uint32_t bytes, uint32_t dst_lo, uint32_t done_now, uint32_t target_prev,
                           uint32_t completed, uint32_t too_small, uint32_t lane) {
    const uint32_t n = count_word & kCountMask;
    // Submissions not yet completed, this one and those on their way included, taken to be as long as this one.
    const uint32_t in_flight = static_cast<uint32_t>(s_k) - completed + 1u + following(count_word);
    uint32_t per_ticket = fixed_per_ticket != 0
                              ? fixed_per_ticket
                              : ticket_size_for_submission(in_flight, n, bytes, workers, (count_word & kBurstEntry) != 0);
    // Small tickets spread a small backlog over many workgroups, at the price of more tickets to write.  When
    // submissions queue up at the leader, its time per submission is what limits the engine, not the spread:
    // a stream of 1 MiB requests of 256 whole pages, 64 in flight, is served at 1.44 M/s in tickets of 8 (which
    // the backlog alone asks for: the workers empty it as fast as it comes), at 1.96 M/s in tickets of 16, and at
    // 1.64 M/s with this rule, which holds for part of the time.
    if (fixed_per_ticket == 0 && per_ticket < too_small) per_ticket = kFullTicket;
    const uint32_t nt = tickets_for(n, per_ticket);
    const uint32_t slot = static_cast<uint32_t>(s_k) & ring_mask;
    // The job slot is free once every ticket ever issued for it has been counted; the ticket ring has room
    // while fewer than its size are outstanding (32-bit wrapping arithmetic).  Otherwise leave this entry
    // for a later poll.
    if (done_now != target_prev && nt != 1) return false;
    if (nt > ticket_room(static_cast<uint32_t>(tickets_out), tickets_done)) return false;
    const uint32_t target = nt == 1 ? target_prev : target_prev + nt;
    if (lane == 0) {
      sys_store_global(&job_target[slot], target);
      if (stamps) sys_store_global(&stamps[kStampsPerJob * slot], clock_now());
    }
    // Four neighbouring lanes write the four sectors of one ticket, so that one store instruction of the
    // wavefront fills 16 consecutive tickets (1 KiB of whole lines).  A ticket's sector differs from the entry's
    // in two places only: `v` is the entry's sector of the lane's own kind.
    // What changes from one pass to the next is kept running, per lane, instead of being worked out from the
    // ticket's index each time (the leader spends three quarters of its time on a stream of 4 MiB requests in
    // this loop and the lines before it).
    const uint32_t sector = lane & 3u;
    const uint32_t first = lane >> 2;
    constexpr uint32_t kPerPass = kWaveLanes / 4;
    // (asked in this order: a request that is alone pays for nothing but the first comparison)
    const bool across = in_flight >= kManyInFlight && shares_across_tickets(in_flight, n, bytes, dst_lo);
    const uint64_t descs = (static_cast<uint64_t>(v.z) << 32) | v.y;  // in the lanes of sector 1: dst_hi, descs
    if (sector == 3) v.z = target;                                     // in the lanes of sector 3: val_hi, n, bytes
    uint64_t d = descs + static_cast<uint64_t>(first) * per_ticket * sizeof(tcpxuLoadMeta);
    const uint64_t d_step = static_cast<uint64_t>(kPerPass) * per_ticket * sizeof(tcpxuLoadMeta);
    uint32_t left = n - first * per_ticket;  // descriptors from this lane's ticket on (meaningless beyond nt)
    uint32_t at = static_cast<uint32_t>(tickets_out) + first;  // low word of the ticket number
    uint8_t* const ring = reinterpret_cast<uint8_t*>(st->tickets) + 16 * sector;
    // The ticket's own word: count | job slot | whether the submission has tickets before and after this one
    // (the last ticket is the one that takes all that is left).
    const uint32_t across_bits = across ? kMoreBefore | kMoreAfter : 0u;
    const uint32_t fixed_bits = (slot << 8) | (nt == 1 ? kOnlyTicket : 0u), after_bit = across_bits & kMoreAfter;
    uint32_t before_bit = first != 0 ? across_bits & kMoreBefore : 0u;
    for (uint32_t i = first; i < nt; i += kPerPass) {
      v.w = at + 1u;  // the stamp
      if (sector == 1) {
        v.y = static_cast<uint32_t>(d);
        v.z = static_cast<uint32_t>(d >> 32);
      }
      if (sector == 3) v.y = std::min(per_ticket, left) | fixed_bits | (left > per_ticket ? after_bit : 0u) | before_bit;
      before_bit = across_bits & kMoreBefore;  // every ticket but the submission's first
      store_vec_sys(ring + static_cast<size_t>(at & (kTicketRing - 1)) * sizeof(Record), v);
      d += d_step;
      left -= kPerPass * per_ticket;
      at += kPerPass;
    }
    lanes_together();
    tickets_out += nt;
    wide = nt > 1 && following(count_word) == 0 ? 1u : 0u;
    return true;
  };
  bool storm_next = false;
  uint32_t storm_backoff = 0, storm_backoff_len = 4;  // polls until the rolling loop is next tried from the several-tickets way
  const bool ring_allows_deep = ring_mask + 1u >= (kDeepGroups + 1) * kPollEntries;
  const bool ring_allows_storm = ring_mask + 1u >= 2 * ((kDeepGroups + 1) * kPollEntries + kStormBacklog);
  // Fixed per-lane roles in the auxiliary load (second load of every poll), so that both loads of a poll are
  // issued back to back by all lanes and waited for once.  What is known of an entry's job slot is in two of the four lanes that
  // hold its sectors, where the other two get at it with one move:
  //   lane 4k     jobs_done of the job slot of entry s+k           lane 4k+1    job_target of the same slot
  //   lane 2      low word of the host stop word                   lane 6       low word of jobs_completed
  //   lane 10     in a deep poll, the stamp of an entry ahead      other lanes repeat lane 2.
  const uint32_t* const host_stop_lo = reinterpret_cast<const uint32_t*>(&ctl->stop);
  const uint32_t* const jobs_completed_lo = reinterpret_cast<const uint32_t*>(&st->jobs_completed.value);

  for (;;) {
    // (Every 64 entries it takes count as one deep poll in this launch's figures.)
    if (storm_next) {
      storm_next = false;
      const StormEnd end = leader_storm(ctl, st, stamps, ring_mask, fixed_per_ticket, s, tickets_out);
      s = same_in_all_lanes(end.s);
      tickets_out = same_in_all_lanes(end.tickets_out);
      const uint32_t taken = same_in_all_lanes32(end.entries);
      entries += taken;
      polls += (taken + (kDeepGroups + 1) * kPollEntries - 1) / ((kDeepGroups + 1) * kPollEntries);
      deep_polls += (taken + (kDeepGroups + 1) * kPollEntries - 1) / ((kDeepGroups + 1) * kPollEntries);
      deep = ring_allows_deep ? 1u : 0u;
      direct = deep;
      // Nothing taken: the queue was not deep, or what waits is not for that loop.  Wait longer each time before
      // asking again (an attempt costs a round trip), and start over once it has worked.
      storm_backoff_len = taken != 0 ? 4u : std::min(2u * storm_backoff_len, 256u);
      storm_backoff = taken != 0 ? 0u : storm_backoff_len;
    } else if (storm_backoff != 0) {
      --storm_backoff;
    }
    if (too_many_out()) ask_done();  // (after the rolling loop, which may have filled the ring)
    // What depends on the lane is worked out afresh in every pass (the empty statement hides from the compiler that
    // the lane is the same each time): a dozen per-lane addresses kept in registers for the life of the loop are
    // what would push the kernel beyond the 80 vector registers that let two workgroups share a compute unit, and a
    // pass waits a microsecond for the host's memory anyway.
    uint32_t lane = threadIdx.x;
    asm volatile("" : "+v"(lane));
    // One round trip fetches entries s .. s+15: lane 4k+j reads sector j (three payload words and the stamp) of
    // entry s+k.
    const uint32_t k_of_lane = lane >> 2;
    const uint8_t* sect_of_lane = reinterpret_cast<const uint8_t*>(&ctl->ring[(s + k_of_lane) & ring_mask]) + 16 * (lane & 3);
    const uint32_t* aux_addr = host_stop_lo;
    const uint32_t kind = lane & 3u;
    auto job_slot_word = [&](uint64_t s0) {  // of the lanes that read one, for the sixteen entries from s0 on
      // (the slots' targets follow their counts in memory)
      return jobs_done + (((static_cast<uint32_t>(s0) + k_of_lane) & ring_mask) + (kind == 1 || s0 + kPollEntries <= free_until ? ring_mask + 1u : 0u));
    };
    if (kind < 2) aux_addr = job_slot_word(s);
    else if (lane == kAuxJobsCompleted) aux_addr = jobs_completed_lo;
    u32x4 sect;
    uint32_t aux;
    uint32_t gone = 0;  // entries of this look's sixteen that an earlier look has brought
    // A deep poll: entries s+16 .. s+63 and their job slots' counters ride along in the same round trip.
    u32x4 sect_more[kDeepGroups];
#pragma unroll
    for (uint32_t g = 0; g < kDeepGroups; ++g) sect_more[g] = u32x4{0u, 0u, 0u, 0u};
    uint32_t aux_more[kDeepGroups] = {};
    if (direct != 0) {
      under_way = 0;  // (what has been asked for lands in LDS and is not looked at)
      ++polls;
      sect = load_vec_sys(sect_of_lane);
      if (deep != 0 && lane == kAuxProbe) aux_addr = &ctl->ring[(s + (kDeepGroups + 1) * kPollEntries + kStormBacklog - 1) & ring_mask].w[15];
      aux = sys_load(aux_addr);
      if (deep != 0) {
        ++deep_polls;
#pragma unroll
        for (uint32_t g = 0; g < kDeepGroups; ++g) {
          const uint64_t s_g = s + (g + 1) * kPollEntries;
          sect_more[g] = load_vec_sys(reinterpret_cast<const uint8_t*>(&ctl->ring[(s_g + k_of_lane) & ring_mask]) + 16 * (lane & 3));
          aux_more[g] = sys_load(job_slot_word(s_g));
        }
      }
      // All of it waited for here: left to the places where it is used, which looks reach as well, the compiler would
      // wait there for what looks have under way.
      asm volatile("" : "+v"(sect), "+v"(aux));
#pragma unroll
      for (uint32_t g = 0; g < kDeepGroups; ++g) asm volatile("" : "+v"(sect_more[g]), "+v"(aux_more[g]));
    } else {
      // Ask for looks from s on until kLooks are under way, then wait for the oldest: a wavefront's vector memory
      // instructions complete in the order issued, and at least kLookLoads for each of the others (stores on top of them)
      // have been issued since its own.
      // Stays here for as long as looks show nothing, entries of one ticket each, few enough for looks, or few of any kind.
      const uint32_t list_of = lane / kCarriedDescs, list_at = lane % kCarriedDescs;  // the four lists, a descriptor to a lane
      const uint8_t* const lists = reinterpret_cast<const uint8_t*>(&ctl->ring[ring_mask + 1u]) + 16 * list_at;
      LdsLook* l = nullptr;
      bool all_taken;
      uint32_t again = 0;  // the look that was gone through last has more to show
#pragma unroll 1
      for (;;) {
        if (again == 0) {
#pragma unroll 1
          while (under_way != kLooks) {
            ask_for_look(&looks[look], aux_addr, lists + ((s + list_of) & ring_mask) * sizeof(CarriedList), sect_of_lane);
            look = same_in_all_lanes32((look + 1u) % kLooks);
            asked_at = same_in_all_lanes64((asked_at << kAskedBits) | (s & kAskedMask));
            under_way = same_in_all_lanes32(under_way + 1u);
          }
          asm volatile("s_waitcnt vmcnt(%0)" : : "n"((kLooks - 1) * kLookLoads) : "memory");
          l = &looks[(look - under_way) % kLooks];
          under_way = same_in_all_lanes32(under_way - 1u);
          ++polls;  // (a look counts when it is gone through, once, whatever becomes of its entries)
          gone = same_in_all_lanes32(static_cast<uint32_t>(s - (asked_at >> (kAskedBits * under_way))) & kAskedMask);
        }
        // Entry s sits `gone` places from the front; what lies beyond the sixteen is not in this look.
        u32x4 sc = *reinterpret_cast<lds_u32x4*>(l->sect[(lane + 4 * gone) % kWaveLanes]);
        const uint32_t word = l->aux[lane];
        u32x4 travels = *reinterpret_cast<lds_u32x4*>(l->carried[(lane + kCarriedDescs * gone) % kWaveLanes]);
        const uint32_t list_count = l->sect[(4 * (list_of + gone) + 3) % kWaveLanes][1];
        const uint32_t completed = lane_value(word, kAuxJobsCompleted);
        const uint64_t there = __ballot(sc.w == static_cast<uint32_t>(s + k_of_lane + 1) && k_of_lane + gone < kPollEntries);
        all_taken = false;
        if ((there & 0xFull) != 0xFull) {  // entry s is not there
          if (lane_value(word, kAuxHostStop) != 0) break;
          if (completed == static_cast<uint32_t>(s)) nothing_under_way();
          if (completed != static_cast<uint32_t>(mirrored)) {
            mirrored = same_in_all_lanes64(mirrored + (completed - static_cast<uint32_t>(mirrored)));
            if (lane == 0) sys_store_global(&ctl->completed, mirrored);
            lanes_together();
          }
          idle = same_in_all_lanes32(idle + 1u);
          if (idle >= idle_limit) break;
          __builtin_amdgcn_s_sleep(kLookSleep);
          continue;
        }
        // The leading entries of one ticket each (sized as ticket_size_for_submission does).
        const uint32_t count = quad_value<3>(sc.y), n = count & kCountMask;
        const uint32_t in_flight = static_cast<uint32_t>(s + k_of_lane + 1) - completed + following(count);
        const uint32_t one_ticket = fixed_per_ticket != 0 ? fixed_per_ticket : in_flight >= kManyInFlight ? kSmallSubmission : kCarriedDescs;
        const uint64_t singles = __ballot(n - 1u < one_ticket) & there;
        auto leading = [](uint64_t m) {
          const uint64_t not_whole = ~(m & (m >> 1) & (m >> 2) & (m >> 3)) & 0x1111111111111111ull;
          return not_whole == 0 ? kPollEntries : static_cast<uint32_t>(__builtin_ctzll(not_whole)) >> 2;
        };
        const uint32_t ready = leading(there);
        uint32_t run = same_in_all_lanes32(std::min(leading(singles), ticket_room(static_cast<uint32_t>(tickets_out), tickets_done)));
        if (run == 0) {
          // One of several tickets, by itself or among few, is handed out here too.
          const uint32_t count_word = lane_value(sc.y, 3);
          if (ready > kFewReady || (count_word & kCountMask) == 0) break;
          const u32x4 own = *reinterpret_cast<lds_u32x4*>(l->sect[4 * gone + (lane & 3u)]);
          if (!write_tickets(s, own, count_word, lane_value(sc.z, 3), lane_value(sc.z, 0), lane_value(word, 4 * gone), lane_value(word, 4 * gone + 1), completed, 0u, lane)) break;
          run = 1;
        } else {
          // The lists that have arrived whole go beside the tickets; the others are fetched by their workgroups.  (A list left beside
          // a ticket's place without the ticket would be taken for that of the one that comes there later.)
          uint32_t bits = 0;
          const uint64_t says_so = __ballot((count & kCarriedEntry) != 0);
          if ((says_so & 0xFFFFull) != 0) {
            const uint32_t list_n = list_count & kCountMask;
            const uint64_t t = tickets_out + list_of;
            const bool list_there = list_at >= list_n || travels.w == static_cast<uint32_t>(s + list_of + 1);
            const bool goes = list_of < run && list_of + gone < kCarriedEntries && (list_count & kCarriedEntry) != 0 && list_n <= kCarriedDescs && static_cast<uint32_t>(t + 1) != 0;
            const uint64_t arrived = __ballot(list_there && goes);
            if (goes && list_at < list_n && ((arrived >> (kCarriedDescs * list_of)) & 0xFFFFull) == 0xFFFFull) {
              travels.w = static_cast<uint32_t>(t + 1);
              store_vec_sys(reinterpret_cast<uint8_t*>(&st->carried[t & (kTicketRing - 1)]) + 16 * list_at, travels);
            }
            lanes_together();
            if (k_of_lane < kCarriedEntries && ((arrived >> (kCarriedDescs * k_of_lane)) & 0xFFFFull) == 0xFFFFull) bits = kCarriedTicket;
          }
          if (k_of_lane < run) {
            const uint64_t t = tickets_out + k_of_lane;
            sc.w = static_cast<uint32_t>(t + 1);
            if ((lane & 3u) == 3) {
              const uint32_t slot = static_cast<uint32_t>(s + k_of_lane) & ring_mask;
              sc.y = n | (slot << 8) | kOnlyTicket | bits;
              if (stamps) sys_store_global(&stamps[kStampsPerJob * slot], clock_now());
            }
            store_vec_sys(reinterpret_cast<uint8_t*>(&st->tickets[t & (kTicketRing - 1)]) + 16 * (lane & 3u), sc);
          }
          lanes_together();
          tickets_out += run;
          wide = 0;
        }
        all_taken = run == ready;
        s = same_in_all_lanes64(s + run);
        tickets_out = same_in_all_lanes64(tickets_out);
        if (lane == 0) sys_store_global(&ctl->head, s);
        lanes_together();
        entries += run;
        idle = 0;
        gone += run;
        deep = same_in_all_lanes32(ring_allows_deep && gone >= kPollEntries ? 1u : 0u);
        direct = same_in_all_lanes32(deep != 0 || run >= kManySmall ? 1u : 0u);
        if ((!all_taken && ready > kFewReady) || direct != 0 || too_many_out()) break;
        again = all_taken ? 0u : 1u;
        sect_of_lane = reinterpret_cast<const uint8_t*>(&ctl->ring[(s + k_of_lane) & ring_mask]) + 16 * (lane & 3);
        if (kind < 2) aux_addr = job_slot_word(s);
      }
      if (all_taken) continue;  // (a poll into registers is next)
      // What stopped the loop is for the rest of this pass, from entry s on.
      sect = *reinterpret_cast<lds_u32x4*>(l->sect[(lane + 4 * gone) & (kWaveLanes - 1)]);
      aux = l->aux[kind < 2 ? (lane + 4 * gone) & (kWaveLanes - 1) : lane];
    }
    // (After the two ways have met: a choice per lane at the end of one of them would make the compiler take everything
    // that differs between them for different from lane to lane.)
    if (k_of_lane + gone >= kPollEntries) sect.w = static_cast<uint32_t>(s + k_of_lane);

    const uint32_t expect = static_cast<uint32_t>(s + k_of_lane + 1);
    const uint64_t ok_mask = __ballot(sect.w == expect);
    // Entries of this poll that are there, counted from the first: lane 4k tells whether all four sectors of entry
    // k are.
    const uint64_t whole = ok_mask & (ok_mask >> 1) & (ok_mask >> 2) & (ok_mask >> 3) & 0x1111111111111111ull;
    const uint64_t missing = ~whole & 0x1111111111111111ull;
    const uint32_t ready = missing != 0 ? static_cast<uint32_t>(__builtin_ctzll(missing)) >> 2 : kPollEntries;
    // The ticket size below which tickets are made 16 instead (see kLeaderBehind; 0: none are).
    const uint32_t too_small = ready >= kLeaderBehind ? kFullTicket : ready >= kLeaderBehindShallow ? kStreamTicket : 0u;
    const uint32_t jobs_completed = lane_value(aux, kAuxJobsCompleted);
    // Payload word i of entry k: component i % 3 of sector i / 3, held by lane 4k + i / 3.
    auto payload_of = [&](uint32_t first_lane, int i) {
      const uint32_t src = first_lane + static_cast<uint32_t>(i / 3);
      return lane_value(i % 3 == 0 ? sect.x : i % 3 == 1 ? sect.y : sect.z, src);
    };

    // Sixteen at a stroke.  The four lanes that hold an entry's sectors hold nearly all of its tickets' words
    // already -- the two records share their layout up to the descriptor pointer and the last sector -- so they
    // write the entry's tickets themselves, ticket i of every entry of the leading run in pass i of one short loop:
    // sixteen submissions of sixteen tickets cost sixteen store instructions, where a pass of the loop below for
    // each (it fetches an entry's words from their lanes into scalars first: about half a microsecond) capped a
    // stream of 1 MiB requests at 2 M/s and a storm of 64 KiB requests at 1.6 M/s.  Taken when the run has some
    // width: a lone entry of many tickets is written faster by the loop below, sixteen tickets to the instruction.
    // (Not for a lone entry that a look shows, which its loop could not write either, nor for one of more descriptors than
    // a ticket holds, nor for a first entry of more than 32 tickets of the size its payload asks for
    // -- 512 whole pages, up to 2048 short fragments: nothing here would apply to them, and what is worked out per lane
    // first would only add to their latency.)
    uint32_t consumed = 0;
    bool deep_next = false;
    const uint32_t n_first = lane_value(sect.y, 3) & kCountMask;
    const uint32_t lane_tickets_hold = kLaneTickets * (fixed_per_ticket != 0 ? fixed_per_ticket : full_ticket_size(lane_value(sect.z, 3), n_first));
    auto view_entries = [&](const u32x4& sc, uint32_t ax, uint64_t s0, uint64_t okm) {
      EntryView v;
      v.n = quad_value<3>(sc.y);      // payload word 10 sits in .y of sector 3
      const uint32_t follow = following(v.n);
      const bool burst = (v.n & kBurstEntry) != 0;
      v.n &= kCountMask;
      v.bytes = quad_value<3>(sc.z);  // payload word 11 sits in .z of sector 3
      const bool all_sectors = ((okm >> (4 * k_of_lane)) & 0xFull) == 0xFull;
      v.target_prev = quad_value<1>(ax);
      v.in_flight = static_cast<uint32_t>(s0 + k_of_lane) - jobs_completed + 1u + follow;
      v.per_ticket = fixed_per_ticket != 0 ? fixed_per_ticket : ticket_size_for_submission(v.in_flight, v.n, v.bytes, workers, burst);
      if (fixed_per_ticket == 0 && v.per_ticket < too_small) v.per_ticket = kFullTicket;  // see below
      v.sane = all_sectors && v.n - 1u < kMaxDescsPerSubmission;  // 1 .. 2^20 descriptors
      v.slot_free = quad_value<0>(ax) == v.target_prev;  // every ticket ever issued for the job slot has been counted
      v.slot = static_cast<uint32_t>(s0 + k_of_lane) & ring_mask;
      return v;
    };
    auto write_single_tickets = [&](const EntryView& v, const u32x4& sc, uint32_t room) {
      return write_single_tickets_of_group(st, stamps, tickets_out, lane, v, sc, room);
    };
    if ((ok_mask & 0xFull) == 0xFull &&  // entry s is there
        ((n_first <= kMaxDescsPerTicket && direct != 0) || (ready >= 2 && n_first <= lane_tickets_hold))) {
      // The groups of sixteen in order (one, or the four of a deep poll), each as long as the one before it went through whole.
      // One loop body that the groups pass through in turn (the registers rotate), so that they are not worked out side by side
      // in as many times the registers: the kernel must stay within 80 for two workgroups per compute unit.
      // (Entries of several tickets go by 64 a round trip as well as those of one, what an entry's four lanes need of each other
      // and of the entries before theirs they get with moves, not by trips through the LDS, and what changes from one ticket to
      // the next is kept running.  Calls of many requests of a few tickets each wait for nothing but this, us before / now: 96 MiB
      // of ragged fragments in requests of 200 KiB 109 / 66, 128 MiB of pages in 300 KiB 96 / 60.6, 100 in 260 87.5 / 53.8, 16 in 260
      // 21.8 / 17.7; with the moves alone 103 and 91, with them and 64 a round trip 71.3, 64.1, 58.0 and 18.4.)
      u32x4 sc = sect, sc1 = sect_more[0], sc2 = sect_more[1], sc3 = sect_more[2];
      uint32_t ax = aux, ax1 = aux_more[0], ax2 = aux_more[1], ax3 = aux_more[2];
      static_assert(kDeepGroups == 3, "the rotation below");
      uint32_t groups = deep != 0 ? kDeepGroups + 1 : 1, several = 0;
      // The first of no more descriptors than one ticket holds: if hundreds more wait, the rolling loop makes one ticket of each
      // such entry (asked once in a while, after sixteen of several tickets).
      const bool may_be_one_each = n_first <= kMaxDescsPerTicket && ring_allows_storm && storm_backoff == 0;
#pragma unroll 1
      for (;;) {
        const uint64_t s_g = s + consumed;
        const uint64_t okm = __ballot(sc.w == static_cast<uint32_t>(s_g + k_of_lane + 1));
        if ((okm & 0xFull) != 0xFull) break;
        const EntryView ev = view_entries(sc, ax, s_g, okm);
        uint32_t run = 0;
        const uint32_t n = ev.n, bytes = ev.bytes, per_ticket = ev.per_ticket, target_prev = ev.target_prev;
        const uint32_t in_flight = ev.in_flight, slot = ev.slot;
        const bool sane = ev.sane, slot_free = ev.slot_free;
        // The ticket ring has room while fewer than its size are outstanding (32-bit wrapping arithmetic).
        const uint32_t room = ticket_room(static_cast<uint32_t>(tickets_out), tickets_done);
        const uint32_t sector = lane & 3u;
        if (__ballot(sane && n > per_ticket) == 0) {
          run = write_single_tickets(ev, sc, room);
          wide = 0;
        } else if (ready >= 2 && lane_value(n, 0) <= kLaneTickets * lane_value(per_ticket, 0)) {
          // Several entries, some of more than one ticket, the first of them not too many.  (The empty statement keeps
          // the compiler from working this block's division and lane exchanges out ahead of the branch, where every
          // poll would pay for them.)
          uint32_t n_here = n, per_here = per_ticket;
          asm volatile("" : "+v"(n_here), "+v"(per_here));
          const uint32_t nt = sane ? tickets_for(n_here, per_here) : 0u;
          const bool regular = sane && nt <= kLaneTickets && (slot_free || nt == 1);
          const uint64_t irregular = ~__ballot(regular);
          const uint32_t run_regular = irregular == 0 ? kPollEntries : static_cast<uint32_t>(__builtin_ctzll(irregular)) >> 2;
          // Tickets of the entries before this one and up to this one (the four lanes of an entry hold the same values).
          const uint32_t mine = k_of_lane < run_regular ? nt : 0u;
          uint32_t upto = mine, most = mine;  // (moves along a row of sixteen lanes, then what the rows before add)
          upto += row_shift<4>(upto);
          upto += row_shift<8>(upto);
          most = std::max(most, row_shift<4>(most));
          most = std::max(most, row_shift<8>(most));
          const uint32_t rows[3] = {lane_value(upto, 15), lane_value(upto, 31), lane_value(upto, 47)};
          upto += (lane >= 16 ? rows[0] : 0u) + (lane >= 32 ? rows[1] : 0u) + (lane >= 48 ? rows[2] : 0u);
          most = std::max(std::max(lane_value(most, 15), lane_value(most, 31)), std::max(lane_value(most, 47), lane_value(most, 63)));
          const uint64_t no_room = ~__ballot(k_of_lane < run_regular && upto <= room);
          const uint32_t fit = no_room == 0 ? kPollEntries : static_cast<uint32_t>(__builtin_ctzll(no_room)) >> 2;
          const uint32_t total = fit != 0 ? lane_value(upto, 4 * fit - 4) : 0u;
          // Taken when the run has some width (`most` is over the regular run, which the room may have cut: an upper
          // bound, good enough for the choice): a lone entry of many tickets is written faster by the loop below.
          if (fit != 0 && total >= 2 * most) {
            const uint32_t target = nt == 1 ? target_prev : target_prev + nt;
            const bool across = shares_across_tickets(in_flight, n, bytes, quad_value<0>(sc.z));  // dst_lo: .z of sector 0
            const bool takes_part = k_of_lane < fit;
            const uint32_t nt_here = takes_part ? nt : 0u;
            // What changes from one ticket to the next is kept running here too (see write_tickets).
            u32x4 v{sc.x, sc.y, sector == 3 ? target : sc.z, 0u};  // in the lanes of sector 1: dst_hi, descs; of sector 3: val_hi, n, bytes
            uint64_t d = (static_cast<uint64_t>(sc.z) << 32) | sc.y;
            uint32_t left = n, at = static_cast<uint32_t>(tickets_out) + (upto - mine), before_bit = 0;
            const uint32_t own_bits = (slot << 8) | (nt == 1 ? kOnlyTicket : 0u);
            for (uint32_t i = 0; i < most; ++i) {
              if (i < nt_here) {
                v.w = at + 1u;  // the stamp
                if (sector == 1) {
                  v.y = static_cast<uint32_t>(d);
                  v.z = static_cast<uint32_t>(d >> 32);
                }
                if (sector == 3) v.y = std::min(per_ticket, left) | own_bits | (across && left > per_ticket ? kMoreAfter : 0u) | before_bit;
                store_vec_sys(reinterpret_cast<uint8_t*>(&st->tickets[at & (kTicketRing - 1)]) + 16 * sector, v);
              }
              before_bit = across ? kMoreBefore : 0u;
              d += per_ticket * sizeof(tcpxuLoadMeta);
              left -= per_ticket;
              ++at;
            }
            if (takes_part && sector == 3) {
              sys_store(&job_target[slot], target);
              if (stamps) sys_store(&stamps[kStampsPerJob * slot], clock_now());
            }
            tickets_out += static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(total)));
            run = same_in_all_lanes32(fit);
            several = 1;
            wide = following(lane_value(sc.y, 4 * run - 1)) == 0 ? 1u : 0u;
          }
        }
        consumed = same_in_all_lanes32(consumed + run);
        if (several != 0 && may_be_one_each) break;
        if (run != kPollEntries || --groups == 0) break;
        sc = sc1, sc1 = sc2, sc2 = sc3;
        ax = ax1, ax1 = ax2, ax2 = ax3;
      }
      deep_next = ring_allows_deep && consumed + gone >= kPollEntries;  // everything that the look could show was there
      // All 64 entries of a deep poll became tickets and the entry kStormBacklog beyond them is published (entries
      // are published in order, so everything up to it is there): a storm, taken from the top of the next pass.  How
      // far the host has got is read off the ring itself: the host's tail word is a line that the host writes with
      // every publish, and a poll that reads it as well waits half a microsecond longer for it.
      if (several != 0) storm_next = may_be_one_each && consumed >= kPollEntries;
      else
        storm_next = ring_allows_storm && consumed == (kDeepGroups + 1) * kPollEntries &&
                     lane_value(aux, kAuxProbe) == static_cast<uint32_t>(s + (kDeepGroups + 1) * kPollEntries + kStormBacklog);
    }
#pragma unroll 1
    for (uint32_t k = consumed; k < kPollEntries; ++k) {
      if (((ok_mask >> (4 * k)) & 0xFull) != 0xFull) break;
      const uint32_t fl = 4 * k;  // first lane of entry k
      const uint32_t count_word = payload_of(fl, 10), n = count_word & kCountMask;
      if (n == 0) {
        const uint32_t flag_lo = payload_of(fl, 6), flag_hi = payload_of(fl, 7);
        const uint32_t val_lo = payload_of(fl, 8), val_hi = payload_of(fl, 9);
        if (lane == 0) {
          sys_store_global(reinterpret_cast<uint64_t*>((static_cast<uint64_t>(flag_hi) << 32) | flag_lo),
                    (static_cast<uint64_t>(val_hi) << 32) | val_lo);
          __hip_atomic_fetch_add(&st->jobs_completed.value, 1ull, __ATOMIC_RELAXED, SYS);
        }
        lanes_together();
      } else {
        const uint32_t holder = fl + (lane & 3u);
        const u32x4 v{bcast(sect.x, holder), bcast(sect.y, holder), bcast(sect.z, holder), 0u};
        if (!write_tickets(s + k, v, count_word, payload_of(fl, 11), payload_of(fl, 2), lane_value(aux, 4 * k), lane_value(aux, 4 * k + 1), jobs_completed, too_small, lane)) break;
      }
      ++consumed;
    }
    deep = same_in_all_lanes32(deep_next ? 1u : 0u);
    // Several entries of several tickets each in one pass, and no more known to be on their way: a stream that keeps the
    // leader busy.  It is served better by a poll that waits until now to ask and so brings more entries, which become
    // tickets at a stroke, than by a look that was asked for a pass ago (1 MiB requests, 64 in flight: 3.4 M/s by looks
    // alone, with some runs at 2.1; 3.57 with this rule, the same with 2 or 4 for the 3).
    // So is whatever brings kManySmall entries or more at a time (forty requests of 128 KiB in short fragments in one call:
    // 19.6 us by looks, 18.9 with 4, 5 or 6 here, 19.5 with 8 or 12; storms of 64 KiB requests with 32 in flight, 7 entries a
    // look: 4.3 M/s by looks and with 6, 4.2 with 4 and 4.1 with 1).
    direct = same_in_all_lanes32(deep_next || consumed >= (wide != 0 ? kManyAtOnce : kManySmall) ? 1u : 0u);
    if (consumed != 0) {
      consumed = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(consumed)));
      s += consumed;
      entries += consumed;
      idle = 0;
      if (lane == 0) sys_store(&ctl->head, s);
      lanes_together();
      continue;
    }

    // Nothing could be consumed this round.
    const bool nothing_there = (ok_mask & 0xFull) != 0xFull;
    if (ask_what_is_done(static_cast<uint32_t>(tickets_out), tickets_done, !nothing_there)) ask_done();
    if (lane_value(aux, kAuxHostStop) != 0 && nothing_there) {
      // Stop requested and entry s not there.  The host wrote its last tail before the stop word, so a tail
      // read now bounds what is still to come.
      uint64_t tail_now = 0;
      if (lane == 0) tail_now = sys_load(&ctl->tail);
      if (s >= same_in_all_lanes64(tail_now)) {  // (lane 0's)
        reason = 1;
        break;
      }
      continue;
    }
    if (jobs_completed != static_cast<uint32_t>(mirrored)) {
      // (the look brings the count's low word; the host is told the whole)
      mirrored += jobs_completed - static_cast<uint32_t>(mirrored);
      if (lane == 0) sys_store(&ctl->completed, mirrored);
      lanes_together();
    }
    if (spin_limit != kNeverIdleOut && nothing_there && ++idle > idle_limit) {
      // Idle for long enough: leave, so that a device-wide synchronize by anybody returns.  The host relaunches
      // the kernel with its next submission.  A submission must not fall between "the leader stopped looking"
      // and "the host thinks the kernel is running": the leader announces that it is leaving, then looks once
      // more; the host publishes, then checks the announcement.  Each side stores before it loads (and PCIe
      // keeps a read behind the posted write issued before it), so at least one of them sees the other.
      if (lane == 0) sys_store(&ctl->exiting, static_cast<uint64_t>(1));
      drain_memory_ops();
      const uint32_t again = sys_load(&ctl->ring[s & ring_mask].w[lane & 15]);
      const bool there = ((lane & 3) == 3 && lane < 16) ? (again == static_cast<uint32_t>(s + 1)) : true;
      if (__all(there)) {
        if (lane == 0) sys_store(&ctl->exiting, static_cast<uint64_t>(0));
        lanes_together();
        idle = 0;
        continue;
      }
      reason = 2;
      break;
    }
    // (leaves the compute unit's issue slots to its copy wavefronts)
    __builtin_amdgcn_s_sleep(kLookSleep);
  }

  // Every ticket written must be visible before any stop word is.
  const uint32_t lane = threadIdx.x;
  drain_memory_ops();
  if (lane == 0) {
    sys_store(&st->sub_head, s);
    sys_store(&st->tickets_out, tickets_out);
    sys_store(&st->exit_reason, reason);
    const uint64_t totals[3] = {sys_load(&st->leader_polls) + polls, sys_load(&st->leader_entries) + entries,
                                sys_load(&st->leader_deep_polls) + deep_polls};
    sys_store(&st->leader_polls, totals[0]);
    sys_store(&st->leader_entries, totals[1]);
    sys_store(&st->leader_deep_polls, totals[2]);
    sys_store(&ctl->leader_polls, totals[0]);
    sys_store(&ctl->leader_entries, totals[1]);
    sys_store(&ctl->leader_deep_polls, totals[2]);
  }
  drain_memory_ops();
  sys_store(&st->stop[lane].value, 1u);
}

// ---- worker -------------------------------------------------------------------------------------------------------
// A lone request waits for every instruction and every trip to the LDS between its ticket and the first load, and between the
// last store and its completion word.  Hence: values of other lanes by moves and masks, not by exchanges through the LDS; the
// load of the descriptors ahead of what is left in the LDS; one word that says whether there is a ticket and what it is; a
// fragment's record waited for once; what tells the fetcher to go on a store, not an addition; and what the last wavefront has
// to say read while its stores are on their way.  (Us, without / with all of these: 64 KiB of pages 7.50 / 7.42, through the plugin
// 6.79 / 6.57, a page 5.73 / 5.50, 1 MiB of wire fragments 9.87 / 9.55, 2048 requests of 64 KiB through the plugin, 16 posted at a time,
// 908 / 890, of which about 1 % gives back what the one load of a ticket's neighbours, below, costs those; streams of 64 KiB
// requests, 1 / 8 / 64 / 256 in flight, 0.170 / 1.338 / 8.72 / 21.6 M/s without, 0.175 / 1.373 / 8.65 / 21.4 with.)
//
// A worker workgroup is kCopyWaves copy wavefronts and one fetcher wavefront.  Towards the end of ticket i the
// fetcher claims a number, polls that ticket's slot, pulls the ticket's descriptors over PCIe and writes their
// records into the other LDS stage; between two tickets the copy wavefronts only meet the fetcher at one barrier.  The copy wavefront
// that finishes a ticket last counts it.
#ifndef TCPXU_ENGINE_COPY_WAVES
#define TCPXU_ENGINE_COPY_WAVES 8
#endif
constexpr uint32_t kCopyWaves = TCPXU_ENGINE_COPY_WAVES;
constexpr uint32_t kEngineThreads = (kCopyWaves + 1) * kWaveLanes;

// What a copy wavefront needs to know about one fragment, worked out by the fetcher: one descriptor per lane, all
// descriptors of a ticket at once, instead of by each copy wavefront from three descriptors per fragment.
constexpr uint32_t kRecSkip = 0, kRecTiny = 1, kRecRounds = 2;
struct alignas(16) RoundRec {
  uint32_t src_lo, src_hi;     // the fragment's first byte
  uint32_t dst_lo, dst_hi;
  uint32_t next_lo, next_hi;   // the next fragment's first source byte (read only if the last line is shared)
  uint32_t start_off, end_off; // FragmentPlan
  uint32_t len;
  uint32_t nvec;
  uint32_t bits;               // head | tail << 8 | share_next << 16 | kind << 24
  uint32_t pad;
};
static_assert(sizeof(RoundRec) == 48, "three 16-byte LDS reads");

// In a staged ticket's word 10 (see copy_ticket), where the descriptors of a ticket of more than kFullTicket never travel.
constexpr uint32_t kRoundsAlone = kCarriedTicket;
static_assert(kCarriedDescs <= kFullTicket, "the bit has another meaning in tickets that bring their descriptors");
constexpr int kTicketWord = 10;  // of a ticket's payload: never zero, since a ticket has descriptors
struct alignas(16) Stage {
  uint32_t payload[kPayloadWords];  // kTicketWord zero: no more tickets
  RoundRec rec[kMaxDescsPerTicket];
};

// The stages live in LDS, and every access says so: through a plain pointer the compiler loses track of that and
// reads the records with flat instructions (a 64-bit address in vector registers each, and slower).
typedef TCPXU_LDS Stage LdsStage;
typedef TCPXU_LDS uint32_t lds_u32;

__device__ __forceinline__ uint64_t lanes_where(bool holds) { return __builtin_amdgcn_ballot_w64(holds); }
__device__ __forceinline__ uint32_t lane_shift(uint32_t v, uint32_t from_lane) {
  return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(static_cast<int>((from_lane & 63u) << 2), static_cast<int>(v)));
}

// Fetcher: look once at the slot of ticket number `ticket` (one 64-byte read, with this workgroup's stop word and, if
// `ask`, the list that may come with the ticket in the same round trip).  Returns 1 and stages the ticket if it is there.  Wave-uniform.
__device__ uint32_t try_fetch_ticket(DevState* st, const uint32_t* stop_word, uint64_t ticket, LdsStage* stage,
                                     uint32_t lane, bool ask, bool* stop_up, uint64_t* stamps) {
  const Record* rec = &st->tickets[ticket & (kTicketRing - 1)];
  const uint32_t expect = static_cast<uint32_t>(ticket + 1);
  uint32_t word = 0;
  if (lane < 16) word = sys_load(&rec->w[lane]);
  else if (lane == 16) word = sys_load(stop_word);
  // (asked for in the same round trip: a ticket that brings its descriptors along is then there whole)
  u32x4 d = {0u, 0u, 0u, 0u};
  if (ask && lane < kCarriedDescs) d = load_vec_sys(reinterpret_cast<const uint8_t*>(&st->carried[ticket & (kTicketRing - 1)]) + 16 * lane);
  *stop_up = lane_value(word, 16) != 0;
  if (~lanes_where(word == expect) & 0x8888u) return 0;
  const uint32_t ticket_bits = lane_value(word, payload_slot(kTicketWord));
  const uint32_t n = ticket_bits & 0xFFu;
  const bool carried = ask && (ticket_bits & kCarriedTicket) != 0;
  if (carried && (~lanes_where(d[3] == expect) & ((1u << n) - 1u)) != 0) return 0;  // its descriptors are still on their way
  const uint64_t fetched_at = stamps ? clock_now() : 0;
  auto word64 = [&](int lo) {
    return (static_cast<uint64_t>(lane_value(word, payload_slot(lo + 1))) << 32) | lane_value(word, payload_slot(lo));
  };
  const uint64_t bounce = word64(0), dst = word64(2), descs_addr = word64(4);
  // One 16-byte descriptor per lane straight from where the submission keeps them (system scope: never a cached
  // copy); lanes past the end repeat the last one and write no record.
  //
  // The descriptor before the ticket's first and the one after its last come with them, where the submission has them (the
  // neighbouring tickets' fetchers look at the same pairs from the other side): lane l then asks for descriptor l - 1, and one
  // move along the lanes puts them where they are worked on.  What bounds the first tickets of a burst is the number of
  // lines that all workers read over PCIe at once, 3.1 ns each where they are a line or two apart (2.3 in longer stretches):
  // a ticket of 32 whose list starts off a line of 128 bytes takes five, and seven while its neighbours were asked for by
  // themselves (on a line, as in the plugin's slots, it takes six both ways).  (Us a call with lists in mapped memory, before / now: 64 MiB of ragged fragments 34.8 / 34.0, 256 MiB 107.5 / 107.1, 16 MiB of wire fragments in requests of
  // 256 KiB 18.5 / 18.2; lists in the GPU's memory as before.  One load for both kinds of ticket: with a load each in two branches
  // small requests, which have no such neighbours, take 1.5 to 3 % longer.)
  const bool more_before = (ticket_bits & kMoreBefore) != 0, more_after = (ticket_bits & kMoreAfter) != 0;
  uint32_t before_len = 0, before_dlo = 0, before_dhi = 0, after_so = 0, after_len = 0, after_dlo = 0, after_dhi = 0;
  const bool outward = more_before || more_after;
  int mine = static_cast<int>(lane < n ? lane : n - 1u);  // a ticket has at least one descriptor
  const int first = more_before ? -1 : 0, last = static_cast<int>(n) - (more_after ? 0 : 1);  // (of those that a ticket with neighbours asks for)
  const bool one_load = outward && n <= kWaveLanes - 2;
  if (one_load) mine = std::min(std::max(static_cast<int>(lane) - 1, first), last);
  if (carried) d[3] = 0;  // (the stamp's place is the high word of the destination offset)
  else d = load_vec_sys(reinterpret_cast<const uint8_t*>(descs_addr) + 16 * mine);
  // The neighbours, where they are more than lanes are left: by themselves, in the same trip.  (Us a call of 64 lists of 2048
  // fragments in tickets of 64, so / with one load of 64 descriptors from the one before on and a second of two.  1 KiB each: lists on
  // a line, where that is ten lines / eleven, 63.5 / 72.3; one descriptor off it, eleven / nine and the long load on lines, 67.9 / 67.2; two, four
  // or seven off, eleven / ten, 67.8 / 70.3.  512 to 1535 bytes: 66.9 / 76.4, 70.7 / 70.9, 70.5 / 74.3.  The empty statement: in other
  // tickets nothing of it is used.)
  u32x4 outer;
  asm volatile("" : "=v"(outer));
  if (outward && !one_load && lane < 2) outer = load_vec_sys(reinterpret_cast<const uint8_t*>(descs_addr) + 16 * (lane == 0 ? first : last));
  // (After the load: a wait for the LDS on the way to it is one that a request waits for.)
  if (lane < 16 && (lane & 3u) != 3) stage->payload[3 * (lane >> 2) + (lane & 3u)] = word;
  if (outward) {  // wave-uniform: a ticket without such neighbours pays nothing here
    auto from_lane = [](uint32_t v, uint32_t src) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(src))); };
    if (one_load) {
      outer = d;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        d[k] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(outer[k]), kDppWaveShiftLeft1, 0xF, 0xF, false));
    }
    if (more_before) before_len = from_lane(outer[1], 0), before_dlo = from_lane(outer[2], 0), before_dhi = from_lane(outer[3], 0);
    if (more_after) {
      const uint32_t at = one_load ? n + 1 : 1;
      after_so = from_lane(outer[0], at), after_len = from_lane(outer[1], at);
      after_dlo = from_lane(outer[2], at), after_dhi = from_lane(outer[3], at);
    }
  }
  const uint32_t so = d[0], len = d[1];
  const uint64_t doff = (static_cast<uint64_t>(d[3]) << 32) | d[2];
  const uint64_t fdst = dst + doff, fsrc = bounce + so;
  uint32_t kind = kRecRounds;
  FragmentPlan plan = {0, len, 0, 0, len >> 4};
  uint64_t next_src = fsrc;
  bool share_next = false;
  // Fragments of whole destination lines (a message of whole pages into an aligned buffer) share none of them and have
  // no edges: what follows would find just that, a quarter of a microsecond later (64 KiB requests of whole pages, 32 in
  // flight: 4.0 M/s without this line, 4.3 with it).  Tickets that are not so work out both sides of every fragment: with
  // the line before taken from what the neighbour found about the line after, one round of lane exchanges less but more
  // branches, 200 requests of 256 KiB in one call took 47.4 us instead of 46.9, 32 of 2 MiB 32.8 instead of 32.4.
  const uint32_t off_line = (static_cast<uint32_t>(fdst) | len) & (kLineBytes - 1);
  const bool off_lines = lanes_where(lane < n && (off_line != 0 || len == 0)) != 0;
  if (lane == 0 && !off_lines && n > kBurstTicket && n <= kShortBurstTicket && (ticket_bits & kOnlyTicket) == 0)
    stage->payload[kTicketWord] = ticket_bits | kRoundsAlone;
  if (off_lines) {
    // The neighbours' descriptors decide which destination lines are shared with them.  A fragment's neighbours are
    // the nearest descriptors of the ticket that are not empty: an empty descriptor between two fragments (a
    // zero-length control message's, a fragment cut to nothing) leaves them back to back in the destination.
    const uint64_t live = lanes_where(lane < n && len != 0);
    const uint64_t below = live & ((1ull << lane) - 1ull);
    const uint64_t above = lane < 63u ? live & ~((2ull << lane) - 1ull) : 0ull;
    const bool prev_inside = below != 0, next_inside = above != 0;
    // Across a ticket's ends only the very first and the very last descriptor have a neighbour, and only one that
    // is not empty: that is the pair the other ticket sees too.
    const bool prev_outside = !prev_inside && lane == 0 && before_len != 0;
    const bool next_outside = !next_inside && lane + 1 == n && after_len != 0;
    const bool has_prev = prev_inside || prev_outside, has_next = next_inside || next_outside;
    const uint32_t prev_lane = prev_inside ? 63u - static_cast<uint32_t>(__builtin_clzll(below)) : lane;
    const uint32_t next_lane = next_inside ? static_cast<uint32_t>(__builtin_ctzll(above)) : lane;
    uint32_t p_len = lane_shift(len, prev_lane), p_dlo = lane_shift(d[2], prev_lane), p_dhi = lane_shift(d[3], prev_lane);
    uint32_t q_len = lane_shift(len, next_lane), q_dlo = lane_shift(d[2], next_lane), q_dhi = lane_shift(d[3], next_lane);
    uint32_t q_so = lane_shift(so, next_lane);
    if (prev_outside) p_len = before_len, p_dlo = before_dlo, p_dhi = before_dhi;
    if (next_outside) q_len = after_len, q_dlo = after_dlo, q_dhi = after_dhi, q_so = after_so;
    const uint64_t p_dst = dst + ((static_cast<uint64_t>(p_dhi) << 32) | p_dlo);
    const uint64_t q_dst = dst + ((static_cast<uint64_t>(q_dhi) << 32) | q_dlo);
    if (len == 0) kind = kRecSkip;
    else if (fragment_is_tiny(reinterpret_cast<const uint8_t*>(fdst), len)) kind = kRecTiny;
    const bool share_prev = kind == kRecRounds && has_prev && shares_line(p_dst, p_len, fdst, len);
    share_next = kind == kRecRounds && has_next && shares_line(fdst, len, q_dst, q_len);
    plan = FragmentPlan{0, 0, 0, 0, 1};
    if (kind == kRecRounds) plan = plan_fragment(fdst, len, share_prev, share_next);
    if (share_next) next_src = bounce + q_so;
  }
  if (lane < n) {
    lds_u32x4* out = reinterpret_cast<lds_u32x4*>(&stage->rec[lane]);
    out[0] = u32x4{static_cast<uint32_t>(fsrc), static_cast<uint32_t>(fsrc >> 32), static_cast<uint32_t>(fdst), static_cast<uint32_t>(fdst >> 32)};
    out[1] = u32x4{static_cast<uint32_t>(next_src), static_cast<uint32_t>(next_src >> 32), plan.start_off, plan.end_off};
    out[2] = u32x4{len, plan.nvec, plan.head | (plan.tail << 8) | (share_next ? 1u << 16 : 0u) | (kind << 24), 0u};
  }
  if (stamps) {
    const uint32_t job = (ticket_bits >> 8) & 0xFFFFu;
    const uint64_t staged_at = clock_now();
    if (lane == 0) {
      __hip_atomic_fetch_min(&stamps[kStampsPerJob * job + 1], fetched_at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_min(&stamps[kStampsPerJob * job + 2], staged_at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  return 1;
}

// Counts a finished ticket (all of its payload is in memory); the last ticket of a submission publishes the
// completion word.
// `flag` and `rest` are the ticket's payload words 4 to 7 and 8 to 11.
__device__ __forceinline__ void retire_ticket(DevState* st, uint32_t* jobs_done, u32x4 flag, u32x4 rest, uint32_t lane, uint64_t* stamps) {
  if (lane == 0) {
    const uint32_t job = (rest[2] >> 8) & 0xFFFFu;
    const uint32_t target = rest[3];
    const uint64_t done_flag = (static_cast<uint64_t>(flag[3]) << 32) | flag[2];
    const uint64_t done_value = (static_cast<uint64_t>(rest[1]) << 32) | rest[0];
    if ((rest[2] & kOnlyTicket) != 0) {
      // The submission's only ticket completes it: tell the caller first, count afterwards (nobody waits for the
      // counts' round trips).  Its job slot has nothing to count.
      if (stamps) sys_store(&stamps[kStampsPerJob * job + 3], clock_now());
      sys_store_global(reinterpret_cast<uint64_t*>(done_flag), done_value);
      __hip_atomic_fetch_add(&st->tickets_done.value, 1ull, __ATOMIC_RELAXED, SYS);
      __hip_atomic_fetch_add(&st->jobs_completed.value, 1ull, __ATOMIC_RELAXED, SYS);
      return;
    }
    const uint32_t count = __hip_atomic_fetch_add(&jobs_done[job], 1u, __ATOMIC_RELAXED, SYS) + 1u;
    __hip_atomic_fetch_add(&st->tickets_done.value, 1ull, __ATOMIC_RELAXED, SYS);
    if (count == target) {
      // Every other ticket's payload was in memory before it was counted, and so is this one's.
      if (stamps) sys_store(&stamps[kStampsPerJob * job + 3], clock_now());
      sys_store_global(reinterpret_cast<uint64_t*>(done_flag), done_value);
      __hip_atomic_fetch_add(&st->jobs_completed.value, 1ull, __ATOMIC_RELAXED, SYS);
    }
  }
}

// Copy wavefront `wave` of kCopyWaves: its run of consecutive fragments of the staged ticket (an eighth of the
// ticket, rounded up), one round (at most 4 KiB) in flight at a time, or two.  A wavefront that writes one contiguous
// stretch of the destination after another measured about 1 % faster end to end than fragments dealt out in turn
// (wave, wave + kCopyWaves, ...).
__device__ __forceinline__ void copy_ticket(const LdsStage* stage, uint32_t ticket_word, uint32_t wave, uint32_t lane, lds_u32* on_last, uint32_t turn) {
  auto uniform = [](uint32_t v) { return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(v)); };
  wave = uniform(wave);
  const uint32_t n = ticket_word & 0xFFu;
  const uint32_t per = (n + kCopyWaves - 1) / kCopyWaves;
  uint32_t j = wave * per < n ? wave * per : n;
  const uint32_t end = j + per < n ? j + per : n;
  // Told once, when the wavefront turns to the last fragment of its share (at once if it has none): the fetcher
  // uses it to start fetching the next ticket.  Every wavefront has a word of its own for that, which all of its lanes write: a
  // counter would cost an addition of one lane, which is a dozen instructions ahead of a lone request's loads.
  auto on_last_fragment = [&] { __hip_atomic_store(on_last, turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  if (j >= end) on_last_fragment();
  uint32_t nvec_left = 0;
  // The next round of the share into `out`, or false when there is none; `prev` is the round before it (read only
  // while a fragment longer than one round goes on).
  auto produce = [&](CopyRound& out, const CopyRound& prev) -> bool {
    if (nvec_left != 0) {
      out = prev;
      out.edges = 0;  // the first round has copied the edge bytes and the shared line
      out.share_next = 0;
      out.src_vec = prev.src_vec + (static_cast<size_t>(prev.nvec) << 4);
      out.dst_vec = prev.dst_vec + (static_cast<size_t>(prev.nvec) << 4);
      out.nvec = nvec_left < kVecPerRound ? nvec_left : kVecPerRound;
      nvec_left -= out.nvec;
      return true;
    }
    while (j < end) {
      const lds_u32x4* words = reinterpret_cast<const lds_u32x4*>(&stage->rec[j]);
      u32x4 w0 = words[0], w1 = words[1], w2 = words[2];
      // One wait for the three, not one each where the compiler first needs it, and ahead of what is added to the LDS next: it
      // answers a wavefront in order.
      asm volatile("" : "+v"(w0), "+v"(w1), "+v"(w2));
      ++j;
      if (j >= end) on_last_fragment();
      const uint32_t bits = uniform(w2[2]);
      const uint32_t kind = bits >> 24;
      if (kind == kRecSkip) continue;
      const uint8_t* src = reinterpret_cast<const uint8_t*>((static_cast<uint64_t>(uniform(w0[1])) << 32) | uniform(w0[0]));
      uint8_t* dst = reinterpret_cast<uint8_t*>((static_cast<uint64_t>(uniform(w0[3])) << 32) | uniform(w0[2]));
      const uint32_t len = uniform(w2[0]);
      if (kind == kRecTiny) {
        copy_tiny_fragment(src, dst, len, lane);
        continue;
      }
      const uint8_t* src_next = reinterpret_cast<const uint8_t*>((static_cast<uint64_t>(uniform(w1[1])) << 32) | uniform(w1[0]));
      out = first_round_of(src, dst, src_next, len, ((bits >> 16) & 1u) != 0, uniform(w1[2]), uniform(w1[3]), bits & 0xFFu,
                           (bits >> 8) & 0xFFu, uniform(w2[1]), lane, &nvec_left);
      return true;
    }
    return false;
  };
  // Two rounds under way at a time -- the second is worked out and asked for while the first one's loads are on their way,
  // and both are waited for together -- in a ticket of more than kFullTicket descriptors (the leader makes those of short
  // fragments, whose rounds leave half of a wavefront's registers empty) and in a request's only ticket, which is waited
  // for.  The other tickets are of whole pages in a stream, where sixteen wavefronts a compute unit with a page each are
  // all that the memory system takes; so are, in tickets of kShortBurstTicket, those of fragments that lie on destination
  // lines, which have next to nothing between their loads and their stores.  (All one at a time / all in pairs: 2048 requests
  // of 64 KiB through the plugin, 16 posted at a time, 1045 / 1000 us, 256 MiB of ragged fragments 114.2 / 107.6, of whole pages
  // 103.9 / 105.7; streams of fragments on lines, 2 KiB in tickets of 32, 5.67 / 5.38 TB/s r+w, 1 KiB in tickets of 64, 5.29 / 5.35;
  // 64 MiB of pages in tickets of 18 31.2 / 30.9 us.)
  const bool pairs = n > kFullTicket || (ticket_word & kOnlyTicket) != 0;
  const bool alone = n > kFullTicket && (ticket_word & kRoundsAlone) != 0;
  CopyRound r, next;
  CopyRegs x, y;
  bool more = produce(r, r);
  while (more) {
    round_load(r, x, lane);
    if (pairs) {
      const bool second = !alone && produce(next, r);
      if (second) round_load(next, y, lane);
      rounds_wait(x, y);
      round_store_loaded(r, x, lane);
      if (second) {
        round_store_loaded(next, y, lane);
        r = next;
      }
      more = (second || alone) && produce(next, r);
      r = next;
    } else {
      round_store(r, x, lane);
      more = produce(next, r);
      r = next;
    }
  }
}

// The compute unit that the calling wavefront runs on, as an odd number; kNoPlace is none's.
constexpr uint32_t kNoPlace = 2;
__device__ __forceinline__ uint32_t compute_unit_here() {
  uint32_t hw, xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  return (hw & 0xFF00u) | ((xcc & 0xFu) << 16) | 1u;  // compute unit, array and engine of one of the eight XCDs
}

__device__ void worker_loop(DevState* st, uint32_t* jobs_done, uint32_t flags, uint64_t* stamps) {
  __shared__ Stage stages[2];
  __shared__ uint32_t s_waves_done;  // copy wavefronts that have finished (and drained) a ticket, running total
  __shared__ uint32_t s_on_last[kCopyWaves];  // of each copy wavefront, the tickets whose last fragment it has turned to
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & (kWaveLanes - 1);
  const uint32_t wave = tid / kWaveLanes;
  if (tid == 0) {
    s_waves_done = 0;
    for (uint32_t w = 0; w < kCopyWaves; ++w) s_on_last[w] = 0;
  }
  __syncthreads();

  if (wave == kCopyWaves) {
    // ---- fetcher ----
    // Each pass stages this workgroup's next ticket (or the exit marker) into the free LDS stage, then meets the
    // copy wavefronts at the barrier.
    //
    // When to claim the next ticket number.  Numbers are served in order, so a number claimed by a workgroup
    // that is still busy keeps its ticket waiting even if other workgroups are idle; a number claimed only when
    // the workgroup is idle leaves the whole pick-up (claim, ticket record, descriptors over PCIe) exposed.  The
    // fetcher claims when every copy wavefront has turned to its last fragment of the current ticket: what is
    // left of the copy then takes about as long as the pick-up, so neither waits for the other.  (flags bit 1
    // clear: claim only when the copy has finished; bit 0 set: claim right away while tickets are queueing up,
    // i.e. the previous ticket was already there at the first look.)
    const uint32_t* stop_word = &st->stop[blockIdx.x % kStopReplicas].value;
    // (Workgroup 0 is the first to be started, and this is the first thing that it does.)
    uint32_t leader_place;
    while ((leader_place = same_in_all_lanes32(sys_load(&st->leader_place))) == 0) __builtin_amdgcn_s_sleep(1);
    const bool beside_leader = leader_place == same_in_all_lanes32(compute_unit_here());
    if (!beside_leader && lane == 0) __hip_atomic_fetch_add(&st->workers_elsewhere, 1u, __ATOMIC_RELAXED, SYS);
    auto not_needed = [&] { return beside_leader && same_in_all_lanes32(sys_load(&st->workers_elsewhere)) >= kEnoughElsewhere; };
    // (The others may be just starting: a few tens of microseconds for them, before a number is claimed that has to be served.)
    for (uint32_t looks = 0; beside_leader && looks < 32 && !not_needed(); ++looks) __builtin_amdgcn_s_sleep(16);
    uint32_t staged = 0;
    bool eager = false;
    const bool allow_eager = (flags & 1u) != 0;
    const bool early = (flags & 2u) != 0;
    auto gate_open = [&](uint32_t tickets) {
      if (!early) return __hip_atomic_load((lds_u32*)&s_waves_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == tickets * kCopyWaves;
      return lanes_where(__hip_atomic_load((lds_u32*)&s_on_last[lane % kCopyWaves], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != tickets) == 0;
    };
    const uint32_t backoff_cap = (flags >> 8) & 0xFFu;
    for (;;) {
      LdsStage* next = (LdsStage*)&stages[staged & 1];
      if (!eager) {
        // Wait for the copy of ticket staged-1 to finish (LDS only: no memory traffic while waiting).
        while (!gate_open(staged)) __builtin_amdgcn_s_sleep(1);
      }
      if (not_needed()) {
        if (lane == 0) next->payload[kTicketWord] = 0;
        __syncthreads();
        break;
      }
      uint64_t t = 0;
      if (lane == 0) t = __hip_atomic_fetch_add(&st->ticket_head.value, 1ull, __ATOMIC_RELAXED, SYS);
      const uint64_t ticket = same_in_all_lanes64(t);
      bool give_up = false, stop_before = false, first_look = true;
      uint32_t backoff = 1, looks = 0;
      for (;;) {
        bool stop_up = false;
        if (try_fetch_ticket(st, stop_word, ticket, next, lane, looks >= kAskAfter, &stop_up, stamps)) {
          eager = first_look && allow_eager;
          break;
        }
        if (stop_before) {
          // The stop word was already up at the previous look and the ticket is still not there: the leader
          // publishes every ticket before any stop word, so it never will be.
          give_up = true;
          if (lane == 0) next->payload[kTicketWord] = 0;
          break;
        }
        stop_before = stop_up;
        first_look = false;
        if (looks < kAskAfter) ++looks;
        if (!stop_before) {
          // Idle: look again soon, but not at once, so that a thousand idle workgroups do not load the memory system that busy
          // ones are using.  (One request alone at random times, mean over 1 to 1024 descriptors: with one sleep between looks
          // 6.09 us, with up to two 6.22, with up to four 6.33, with a quarter of one 6.06; storms, bursts and streams the same.
          // Another kernel beside the idle engine, with one / two: a copy of 1 GiB 566 / 562 us, of the same 8 MiB 7.3 / 7.2, a gather of
          // 64 MiB 343 / 342.)
          for (uint32_t i = 0; i < backoff; ++i) __builtin_amdgcn_s_sleep(4);
          if (backoff < backoff_cap) backoff <<= 1;
        }
      }
      __syncthreads();  // hands `next` to the copy wavefronts, which are waiting here after their ticket
      if (give_up) break;
      ++staged;
    }
  } else {
    // ---- copy wavefronts ----
    for (uint32_t i = 0;; ++i) {
      __syncthreads();  // stage i&1 is ready
      LdsStage* stage = (LdsStage*)&stages[i & 1];
      const uint32_t ticket_word = same_in_all_lanes32(stage->payload[kTicketWord]);
      if (ticket_word == 0) break;
      copy_ticket(stage, ticket_word, wave, lane, (lds_u32*)&s_on_last[wave], i + 1);
      // (What the last wavefront needs, read while the stores are on their way.)
      const lds_u32x4* words = reinterpret_cast<const lds_u32x4*>(&stage->payload[0]);
      u32x4 flag = words[1], rest = words[2];
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : "+v"(flag), "+v"(rest) : : "memory");  // this wavefront's write-through stores are acknowledged
      uint32_t arrived = 0;
      if (lane == 0)
        arrived = __builtin_amdgcn_atomic_inc32((lds_u32*)&s_waves_done, 0xFFFFFFFFu, __ATOMIC_RELAXED, "workgroup") + 1u;
      // The wavefront that finishes last counts the ticket: every wavefront's payload is in memory by then.
      if (same_in_all_lanes32(arrived) == (i + 1) * kCopyWaves) retire_ticket(st, jobs_done, flag, rest, lane, stamps);
    }
  }
}

__global__ __launch_bounds__(kEngineThreads) __attribute__((amdgpu_waves_per_eu(6))) void unpack_engine_kernel(HostCtl* ctl, DevState* st, uint32_t* jobs_done,
                                                                   uint32_t* job_target, uint32_t ring_mask,
                                                                   uint32_t per_ticket, uint32_t spin_limit,
                                                                   uint32_t flags, uint64_t* stamps) {
  if (blockIdx.x == 0) {
    __shared__ Look looks[kLooks];
    if (threadIdx.x == 0) sys_store_global(&st->leader_place, enough_can_be_elsewhere(gridDim.x) ? compute_unit_here() : kNoPlace);
    if (threadIdx.x < kWaveLanes)
      leader_loop(ctl, st, jobs_done, job_target, ring_mask, per_ticket, spin_limit, stamps, (LdsLook*)&looks[0]);
  } else {
    worker_loop(st, jobs_done, flags, stamps);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    drain_memory_ops();
    const uint32_t before = __hip_atomic_fetch_add(&st->exited_wgs, 1u, __ATOMIC_RELAXED, SYS);
    if (before + 1 == gridDim.x) {
      // Last workgroup out: every ticket that was written has been counted.  Ticket numbers claimed beyond the
      // last written one are given back, so the next launch starts where this one ended.
      sys_store(&st->ticket_head.value, sys_load(&st->tickets_out));
      sys_store(&ctl->completed, sys_load(&st->jobs_completed.value));
      drain_memory_ops();
      sys_store(&ctl->exited, static_cast<uint64_t>(sys_load(&st->exit_reason)));
    }
  }
}

}  // namespace
}  // namespace tcpxu

using namespace tcpxu;

struct tcpxuEngine {
  int device = 0;
  uint32_t ring_entries = 0;
  uint32_t workgroups = 0;
  uint32_t per_ticket = 0;
  uint32_t spin_limit = 0;
  uint32_t flags = 0;  // bits 0-1: when fetchers claim (see worker_loop); bits 8-15: idle poll backoff cap
  hipStream_t stream = nullptr;
  hipEvent_t ev_start = nullptr, ev_stop = nullptr;
  HostCtl* ctl = nullptr;      // host address of the mapped control block
  HostCtl* ctl_dev = nullptr;  // its device alias
  DevState* st = nullptr;
  uint32_t* jobs_done = nullptr;   // [ring_entries], device memory
  uint32_t* job_target = nullptr;  // [ring_entries], device memory, leader-private
  uint64_t tail = 0;  // host copy
  uint64_t head_seen = 0;  // the leader's position as last read
  bool launched = false;  // between a launch and the Stop that reaps it (the kernel may have left by itself)
  bool failed = false;    // the kernel stopped answering (see tcpxuEngineSubmitSized); nothing more is accepted
  uint64_t launches = 0;
  uint64_t submissions = 0;
  MappedView mapped;           // what mapped host memory there is (see carry_descriptors)
  uint64_t* stamps = nullptr;  // device memory, kStampsPerJob per ring entry, or null (tcpxuEngineEnableStamps)
  std::mutex mu;
};

static size_t ctl_bytes(uint32_t ring_entries) {
  return offsetof(HostCtl, ring) + (sizeof(Record) + sizeof(CarriedList)) * ring_entries;
}

extern "C" {

int tcpxuEngineCreate(int device, const tcpxuEngineConfig* config, tcpxuEngine** engine) {
  if (!engine) return TCPXU_INVALID_ARGUMENT;
  *engine = nullptr;
  tcpxuEngineConfig cfg{};
  if (config) cfg = *config;
  if (cfg.ring_entries == 0) cfg.ring_entries = 4096;
  if ((cfg.ring_entries & (cfg.ring_entries - 1)) != 0 || cfg.ring_entries > (1u << 16) || cfg.ring_entries < kSmallestRing) {
    set_error("ring_entries %u must be a power of two in [%u, 65536]", cfg.ring_entries, kSmallestRing);
    return TCPXU_INVALID_ARGUMENT;
  }
  if (cfg.descs_per_ticket == 0) {
    const char* v = getenv("TCPXU_DESCS_PER_TICKET");  // tuning aid: fixes the size; unset = by backlog
    if (v && *v) cfg.descs_per_ticket = static_cast<uint32_t>(atoi(v));
  }
  if (cfg.descs_per_ticket > kMaxDescsPerTicket) {
    set_error("descs_per_ticket %u must be in [0,%u]", cfg.descs_per_ticket, kMaxDescsPerTicket);
    return TCPXU_INVALID_ARGUMENT;
  }
  DeviceScope scope(device);
  TCPXU_TRY(scope.rc());
  const uint32_t cus = static_cast<uint32_t>(std::max(1, device_compute_units(device)));
  if (cfg.workgroups == 0) {
    // Two worker workgroups per compute unit: 18 of a compute unit's 32 wavefront slots, so that other kernels
    // (copies, the caller's own work) are scheduled beside the engine while it runs.  One is not enough (8 MiB
    // chunks, 64 slots in flight: 59 % of the HBM roofline against 71 %; fragments of 2 KiB: 41 % against 66 %).
    // Two is also all that is ever resident: the nine wavefronts of a workgroup go to the four SIMDs as 3+2+2+2,
    // a third workgroup would need a ninth slot on the first SIMD, and the hardware counters show a grid of
    // three per compute unit running exactly the wavefront-cycles of two.  (Workgroups of twelve wavefronts, two
    // per compute unit, do fit: 22 copy wavefronts instead of 16 move short fragments 1 % faster and whole pages
    // no faster, and leave other kernels 8 slots instead of 14.)  The occupancy query is not asked: it has answered
    // "one" in a process that had launched other kernels before.  A grid larger than what is resident would still
    // be correct -- no workgroup waits for another worker -- only pointless.
    uint32_t per_cu = 2;
    const char* v = getenv("TCPXU_ENGINE_WGS_PER_CU");  // tuning aid: 1 or 2
    if (v && *v) per_cu = std::min(std::max(static_cast<uint32_t>(atoi(v)), 1u), 2u);
    cfg.workgroups = cus * per_cu + 1;
  }
  if (cfg.workgroups < 2 || cfg.workgroups > (1u << 16)) {
    set_error("an engine needs the leader workgroup and 1 to 65535 workers");
    return TCPXU_INVALID_ARGUMENT;
  }

  tcpxuEngine* e = new (std::nothrow) tcpxuEngine;
  if (!e) return TCPXU_SYSTEM_ERROR;
  e->device = device;
  e->ring_entries = cfg.ring_entries;
  e->workgroups = cfg.workgroups;
  e->per_ticket = cfg.descs_per_ticket;
  e->spin_limit = cfg.spin_limit != 0 ? cfg.spin_limit : kDefaultIdlePolls;
  {
    const char* ve = getenv("TCPXU_ENGINE_EAGER");
    const char* vb = getenv("TCPXU_ENGINE_BACKOFF_CAP");
    const uint32_t eager = (ve && *ve) ? static_cast<uint32_t>(atoi(ve)) & 3u : 2u;
    const uint32_t cap = (vb && *vb) ? static_cast<uint32_t>(atoi(vb)) & 0xFFu : 1u;
    e->flags = eager | (cap << 8);
  }
  int rc = TCPXU_SUCCESS;
  do {
    void *h = nullptr, *d = nullptr;
    if ((rc = tcpxuMappedAlloc(device, ctl_bytes(cfg.ring_entries), &h, &d)) != TCPXU_SUCCESS) break;
    e->ctl = static_cast<HostCtl*>(h);
    e->ctl_dev = static_cast<HostCtl*>(d);
    const size_t st_bytes = sizeof(DevState) + 2 * sizeof(uint32_t) * cfg.ring_entries;
    // The state is cleared on the engine's own stream, and an event pair goes through it, so that whatever the
    // runtime sets up at a stream's first use (its hardware queue: half a millisecond) is paid here and not by the
    // first request.
    // Asking for the kernel's attributes makes the runtime load its code now (lazy otherwise: the first launch
    // would spend half a millisecond on it, after the launch's start event has been recorded).
    hipFuncAttributes attr;
    if (hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(unpack_engine_kernel)) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&e->st), st_bytes) != hipSuccess ||
        hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&e->ev_start) != hipSuccess || hipEventCreate(&e->ev_stop) != hipSuccess ||
        hipEventRecord(e->ev_start, e->stream) != hipSuccess ||
        hipMemsetAsync(e->st, 0, st_bytes, e->stream) != hipSuccess ||
        hipEventRecord(e->ev_stop, e->stream) != hipSuccess || hipStreamSynchronize(e->stream) != hipSuccess ||
        hipDeviceSynchronize() != hipSuccess) {
      set_error("engine allocation failed: %s", hipGetErrorString(hipGetLastError()));
      rc = TCPXU_DEVICE_ERROR;
      break;
    }
    e->jobs_done = reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(e->st) + sizeof(DevState));
    e->job_target = e->jobs_done + cfg.ring_entries;  // (leader_loop's job_slot_word finds the second by the first)
    // Test aid: where the engine's counts of submissions and tickets start.  Records are stamped with the low 32 bits
    // of their sequence number, and a busy engine passes 2^32 submissions within the hour; a test that starts just
    // below sees the crossing in milliseconds.  (Start more than a lap of the ticket ring below: a slot of either ring
    // that was never written reads as stamped for sequence number 2^32-1, which an engine that counts from zero
    // reaches only after every slot has been written many times.)
    const char* vc = getenv("TCPXU_ENGINE_COUNT_FROM");
    if (vc && *vc) {
      const uint64_t from = strtoull(vc, nullptr, 0);
      const uint32_t to_wrap = 0u - static_cast<uint32_t>(from);
      if (to_wrap != 0 && to_wrap <= std::max(kTicketRing, e->ring_entries)) {
        set_error("TCPXU_ENGINE_COUNT_FROM: %u is less than a lap of the rings below 2^32", to_wrap);
        rc = TCPXU_INVALID_ARGUMENT;
        break;
      }
      uint64_t* const counts[] = {&e->st->ticket_head.value, &e->st->tickets_done.value, &e->st->jobs_completed.value, &e->st->sub_head,
                                  &e->st->tickets_out};  // device addresses: only computed here, never read
      for (uint64_t* c : counts) {
        if (hipMemcpy(c, &from, sizeof from, hipMemcpyHostToDevice) != hipSuccess) {
          set_error("engine counters: %s", hipGetErrorString(hipGetLastError()));
          rc = TCPXU_DEVICE_ERROR;
          break;
        }
      }
      e->tail = e->head_seen = from;
      e->ctl->tail = e->ctl->head = e->ctl->completed = from;
    }
  } while (false);
  if (rc != TCPXU_SUCCESS) {
    tcpxuEngineDestroy(e);
    return rc;
  }
  *engine = e;
  return TCPXU_SUCCESS;
}

// Launches the kernel.  Caller holds e->mu; any previous launch has ended (its exit word is set).
static int launch_locked(tcpxuEngine* e) {
  DeviceScope scope(e->device);
  TCPXU_TRY(scope.rc());
  // Per-launch state: exit bookkeeping and stop words start from zero; positions and counters are kept.
  TCPXU_HIP(hipMemsetAsync(reinterpret_cast<uint8_t*>(e->st) + offsetof(DevState, exited_wgs), 0,
                           offsetof(DevState, tickets) - offsetof(DevState, exited_wgs), e->stream));
  std::atomic_thread_fence(std::memory_order_seq_cst);
  e->ctl->stop = 0;
  e->ctl->exited = 0;
  e->ctl->exiting = 0;
  std::atomic_thread_fence(std::memory_order_seq_cst);
  TCPXU_HIP(hipEventRecord(e->ev_start, e->stream));
  hipLaunchKernelGGL(unpack_engine_kernel, dim3(e->workgroups), dim3(kEngineThreads), 0, e->stream, e->ctl_dev, e->st,
                     e->jobs_done, e->job_target, e->ring_entries - 1, e->per_ticket, e->spin_limit, e->flags, e->stamps);
  TCPXU_HIP(hipGetLastError());
  TCPXU_HIP(hipEventRecord(e->ev_stop, e->stream));
  e->launched = true;
  e->launches += 1;
  return TCPXU_SUCCESS;
}

static uint64_t host_load(const uint64_t* p) {
  return reinterpret_cast<const std::atomic<uint64_t>*>(p)->load(std::memory_order_acquire);
}

int tcpxuEngineStart(tcpxuEngine* e) {
  if (!e) return TCPXU_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(e->mu);
  if (e->launched && host_load(&e->ctl->exited) == 0) {
    set_error("engine already started");
    return TCPXU_INVALID_USAGE;
  }
  return launch_locked(e);
}

int tcpxuEngineStop(tcpxuEngine* e, double* elapsed_us) {
  if (!e) return TCPXU_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(e->mu);
  if (!e->launched) {
    set_error("engine is not started");
    return TCPXU_INVALID_USAGE;
  }
  DeviceScope scope(e->device);
  TCPXU_TRY(scope.rc());
  std::atomic_thread_fence(std::memory_order_seq_cst);
  reinterpret_cast<std::atomic<uint64_t>*>(&e->ctl->stop)->store(1, std::memory_order_seq_cst);
  // Wait for the kernel's own exit word first, with a deadline: a stuck kernel then surfaces as an error
  // from this call instead of a host thread parked inside the runtime.
  const char* v = getenv("TCPXU_ENGINE_STOP_TIMEOUT_MS");
  const long timeout_ms = (v && *v) ? atol(v) : 20000;
  const auto t0 = std::chrono::steady_clock::now();
  while (reinterpret_cast<std::atomic<uint64_t>*>(&e->ctl->exited)->load(std::memory_order_acquire) == 0) {
    if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(timeout_ms)) {
      set_error("engine kernel did not exit within %ld ms of the stop request", timeout_ms);
      return TCPXU_INTERNAL_ERROR;
    }
    std::this_thread::yield();
  }
  TCPXU_HIP(hipEventSynchronize(e->ev_stop));
  if (elapsed_us) {
    float ms = 0.f;
    TCPXU_HIP(hipEventElapsedTime(&ms, e->ev_start, e->ev_stop));
    *elapsed_us = static_cast<double>(ms) * 1000.0;
  }
  e->launched = false;
  return TCPXU_SUCCESS;
}

int tcpxuEngineDestroy(tcpxuEngine* e) {
  if (!e) return TCPXU_SUCCESS;
  if (e->launched) {
    int rc = tcpxuEngineStop(e, nullptr);
    if (rc != TCPXU_SUCCESS) return rc;  // never free memory under a running kernel
  }
  DeviceScope scope(e->device);
  if (e->ev_start) (void)hipEventDestroy(e->ev_start);
  if (e->ev_stop) (void)hipEventDestroy(e->ev_stop);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  if (e->st) (void)hipFree(e->st);
  if (e->stamps) (void)hipFree(e->stamps);
  if (e->ctl) (void)tcpxuMappedFree(e->device, e->ctl);
  delete e;
  return TCPXU_SUCCESS;
}

int tcpxuEngineSubmit(tcpxuEngine* e, const void* bounce_base, void* dst_base, const void* descs_dev,
                      uint32_t n_descs, void* done_flag_dev, uint64_t done_value) {
  return tcpxuEngineSubmitSized(e, bounce_base, dst_base, descs_dev, n_descs, 0, done_flag_dev, done_value);
}

int tcpxuEngineSubmitSized(tcpxuEngine* e, const void* bounce_base, void* dst_base, const void* descs_dev,
                           uint32_t n_descs, uint64_t payload_bytes, void* done_flag_dev, uint64_t done_value) {
  const tcpxuSubmission one = {bounce_base, dst_base, descs_dev, done_flag_dev, done_value, n_descs,
                               payload_bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : static_cast<uint32_t>(payload_bytes)};
  uint32_t accepted = 0;
  return tcpxuEngineSubmitMany(e, &one, 1, &accepted);
}

// What a submission must look like; decided on the host, before anything is queued.
static int check_submission(const tcpxuEngine* e, const tcpxuSubmission& s) {
  if (!s.done_flag_dev || s.done_value == 0 || reinterpret_cast<uintptr_t>(s.done_flag_dev) % 8 != 0) {
    set_error("submit needs an 8-byte aligned completion word and a nonzero completion value");
    return TCPXU_INVALID_ARGUMENT;
  }
  if (s.n_descs > 0 && (!s.bounce_base || !s.dst_base || !s.descs_dev || reinterpret_cast<uintptr_t>(s.descs_dev) % 16 != 0)) {
    set_error("submit needs bounce, destination and a 16-byte aligned descriptor address");
    return TCPXU_INVALID_ARGUMENT;
  }
  // A submission whose tickets can never all fit the ticket ring would sit at the head of the submission ring for
  // ever, and the leader neither stops nor idles out with an entry waiting.
  if (s.n_descs > max_descs_for(e->per_ticket)) {
    set_error("%u descriptors in one submission exceed the limit of %u (tickets of %u at least, %u tickets in flight at most)",
              s.n_descs, max_descs_for(e->per_ticket), e->per_ticket ? e->per_ticket : kSmallestAdaptiveTicket, kTicketRing);
    return TCPXU_INVALID_ARGUMENT;
  }
  return TCPXU_SUCCESS;
}

// Copies a small list's descriptors beside the ring's entry, if they lie in memory that tcpxuMappedAlloc gave out (where
// the host has them too) and their destination offsets fit.  Caller holds e->mu.
static bool carry_descriptors(tcpxuEngine* e, const tcpxuSubmission& sub, uint32_t stamp) {
  const tcpxuLoadMeta* from = static_cast<const tcpxuLoadMeta*>(mapped_host_address(&e->mapped, sub.descs_dev, sizeof(tcpxuLoadMeta) * sub.n_descs));
  if (!from) return false;
  CarriedList* lists = reinterpret_cast<CarriedList*>(&e->ctl->ring[e->ring_entries]);
  CarriedList* list = &lists[e->tail & (e->ring_entries - 1)];
  uint64_t high = 0;
  for (uint32_t i = 0; i < sub.n_descs; ++i) {
    const tcpxuLoadMeta d = from[i];
    high |= d.dst_off >> 32;
    typedef uint32_t host_u32x4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<volatile host_u32x4*>(list->w[i]) = host_u32x4{d.src_off, d.len, static_cast<uint32_t>(d.dst_off), stamp};
  }
  return high == 0;
}

int tcpxuEngineSubmitMany(tcpxuEngine* e, const tcpxuSubmission* subs, uint32_t n, uint32_t* accepted) {
  if (accepted) *accepted = 0;
  if (!e || (!subs && n != 0)) {
    set_error("submit needs an engine and submissions");
    return TCPXU_INVALID_ARGUMENT;
  }
  for (uint32_t i = 0; i < n; ++i) TCPXU_TRY(check_submission(e, subs[i]));  // all or nothing: none is queued if one is refused
  if (n == 0) return TCPXU_SUCCESS;
  std::lock_guard<std::mutex> lock(e->mu);
  if (e->failed) {
    set_error("the engine stopped answering earlier and accepts nothing more");
    return TCPXU_INTERNAL_ERROR;
  }
  // (The leader writes its position into the host's memory with all that it takes, and a line that the GPU has written costs a
  // call a trip to DRAM.  What fits between the last position read and kCarryBehind entries on fits the smallest ring, and the
  // leader is no further behind than that.  Requests of 1 / 4 / 8 / 16 pages through the plugin, 16 posted at a time, us a
  // request: 0.413 / 0.59 / 0.428 / 0.468 with a look in every call, 0.394 / 0.53 / 0.404 / 0.444 with one in sixteen.)
  uint64_t head = e->head_seen;
  if (e->tail + n - head > kCarryBehind) head = e->head_seen = host_load(&e->ctl->head);
  const uint64_t room = e->ring_entries - (e->tail - head);
  const uint32_t take = static_cast<uint32_t>(std::min<uint64_t>(room, n));
  if (take == 0) return kTcpxuInProgress;
  const uint32_t workers = e->workgroups - 1;
  // Submissions before this call's that are not completed, as far as the leader has said (it does with every look that finds
  // nothing new): read only where it is asked for, since it is a line that the GPU writes.  (The leader may have taken and
  // finished entries of this very call by then.)
  const uint64_t tail_before = e->tail;
  uint64_t ahead = UINT64_MAX;
  auto few_ahead = [&](uint32_t n_descs) {
    if (ahead == UINT64_MAX) {
      const uint64_t completed = host_load(&e->ctl->completed);
      ahead = tail_before > completed ? tail_before - completed : 0;
    }
    return few_ahead_of_burst(ahead, n_descs, workers);
  };
  for (uint32_t k = 0; k < take; ++k) {
    const tcpxuSubmission& sub = subs[k];
    const uint64_t v[5] = {reinterpret_cast<uint64_t>(sub.bounce_base), reinterpret_cast<uint64_t>(sub.dst_base),
                           reinterpret_cast<uint64_t>(sub.descs_dev), reinterpret_cast<uint64_t>(sub.done_flag_dev),
                           sub.done_value};
    // The entry's sixteen words in the order they lie (three payload words and the stamp per sector), written as
    // four 16-byte stores: a record is valid for the leader once all four stamps are there, in whatever order the
    // sectors arrive, so nothing has to be ordered within it.
    const uint32_t stamp = static_cast<uint32_t>(e->tail + 1);
    alignas(64) uint32_t w[16];
    uint32_t p[kPayloadWords];
    for (int i = 0; i < 5; ++i) {
      p[2 * i] = static_cast<uint32_t>(v[i]);
      p[2 * i + 1] = static_cast<uint32_t>(v[i] >> 32);
    }
    const bool pages = full_ticket_size(sub.payload_bytes, sub.n_descs) == kFullTicket;
    const bool burst = burst_of_pages(take, sub.n_descs, sub.payload_bytes, workers) ||
                       (burst_of_short_fragments(take, sub.n_descs, sub.payload_bytes, workers) && few_ahead(sub.n_descs));
    p[10] = sub.n_descs | (pages ? 0u : std::min(take - 1 - k, kMostFollow) << kFollowShift) | (burst ? kBurstEntry : 0u);
    p[11] = sub.payload_bytes;
    if (k < kCarriedEntries && sub.n_descs != 0 && sub.n_descs <= kCarriedDescs && stamp != 0 && e->tail - head < kCarryBehind &&
        carry_descriptors(e, sub, stamp))
      p[10] |= kCarriedEntry;
    for (int sct = 0; sct < 4; ++sct) {
      w[4 * sct] = p[3 * sct];
      w[4 * sct + 1] = p[3 * sct + 1];
      w[4 * sct + 2] = p[3 * sct + 2];
      w[4 * sct + 3] = stamp;
    }
    Record* ent = &e->ctl->ring[e->tail & (e->ring_entries - 1)];
    // What the descriptors say must be in memory before the entry that points to them can be seen.
    std::atomic_thread_fence(std::memory_order_release);
    typedef uint32_t host_u32x4 __attribute__((ext_vector_type(4)));
    for (int sct = 0; sct < 4; ++sct)
      *reinterpret_cast<volatile host_u32x4*>(&ent->w[4 * sct]) = *reinterpret_cast<const host_u32x4*>(&w[4 * sct]);
    e->tail += 1;
  }
  e->submissions += take;
  std::atomic_thread_fence(std::memory_order_release);
  reinterpret_cast<std::atomic<uint64_t>*>(&e->ctl->tail)->store(e->tail, std::memory_order_release);
  if (accepted) *accepted = take;
  // The kernel may have left for idleness, or be leaving right now (see leader_loop): publish first, then look.
  if (e->launched) {
    std::atomic_thread_fence(std::memory_order_seq_cst);
    if (host_load(&e->ctl->exiting) != 0 && host_load(&e->ctl->exited) == 0) {
      const auto t0 = std::chrono::steady_clock::now();
      while (host_load(&e->ctl->exiting) != 0 && host_load(&e->ctl->exited) == 0) {
        if (std::chrono::steady_clock::now() - t0 > std::chrono::seconds(5)) {
          // The entries are in the ring and stay there: this is not "not submitted, try again".  The engine is
          // marked failed so that the caller cannot queue the same work twice by retrying.
          e->failed = true;
          set_error("engine kernel announced that it is leaving and never did; the submission stays queued and the "
                    "engine accepts nothing more");
          return TCPXU_INTERNAL_ERROR;
        }
      }
    }
    if (host_load(&e->ctl->exited) == 2) TCPXU_TRY(launch_locked(e));  // it left by itself: bring it back
  }
  return take == n ? TCPXU_SUCCESS : kTcpxuInProgress;
}

int tcpxuEngineEnableStamps(tcpxuEngine* e, double* ticks_per_us) {
  if (!e) return TCPXU_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(e->mu);
  if (e->launched) {
    set_error("stamps are switched on while the engine is stopped");
    return TCPXU_INVALID_USAGE;
  }
  DeviceScope scope(e->device);
  TCPXU_TRY(scope.rc());
  const size_t bytes = sizeof(uint64_t) * kStampsPerJob * e->ring_entries;
  if (!e->stamps) TCPXU_HIP(hipMalloc(reinterpret_cast<void**>(&e->stamps), bytes));
  TCPXU_HIP(hipMemset(e->stamps, 0xFF, bytes));
  if (ticks_per_us) {
    int khz = 0;
    TCPXU_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, e->device));
    *ticks_per_us = khz / 1000.0;
  }
  return TCPXU_SUCCESS;
}

int tcpxuEngineReadStamps(tcpxuEngine* e, uint64_t first_submission, uint32_t n, uint64_t* out) {
  if (!e || !out || n > e->ring_entries) {
    set_error("stamps: at most ring_entries submissions at a time");
    return TCPXU_INVALID_ARGUMENT;
  }
  std::lock_guard<std::mutex> lock(e->mu);
  if (!e->stamps || e->launched) {
    set_error("stamps are read while the engine is stopped, after tcpxuEngineEnableStamps");
    return TCPXU_INVALID_USAGE;
  }
  DeviceScope scope(e->device);
  TCPXU_TRY(scope.rc());
  std::vector<uint64_t> all(static_cast<size_t>(kStampsPerJob) * e->ring_entries);
  TCPXU_HIP(hipMemcpy(all.data(), e->stamps, all.size() * sizeof(uint64_t), hipMemcpyDeviceToHost));
  for (uint32_t i = 0; i < n; ++i) {
    const size_t slot = (first_submission + i) & (e->ring_entries - 1);
    for (uint32_t k = 0; k < kStampsPerJob; ++k) out[kStampsPerJob * i + k] = all[kStampsPerJob * slot + k];
  }
  TCPXU_HIP(hipMemset(e->stamps, 0xFF, all.size() * sizeof(uint64_t)));  // the minima start from ones again
  return TCPXU_SUCCESS;
}

int tcpxuEngineGetStats(tcpxuEngine* e, tcpxuEngineStats* stats) {
  if (!e || !stats) return TCPXU_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(e->mu);
  stats->launches = e->launches;
  stats->submissions = e->submissions;
  stats->leader_polls = host_load(&e->ctl->leader_polls);
  stats->leader_entries = host_load(&e->ctl->leader_entries);
  stats->leader_deep_polls = host_load(&e->ctl->leader_deep_polls);
  return TCPXU_SUCCESS;
}

int tcpxuEngineCompleted(tcpxuEngine* e, uint64_t* completed) {
  if (!e || !completed) return TCPXU_INVALID_ARGUMENT;
  *completed = reinterpret_cast<std::atomic<uint64_t>*>(&e->ctl->completed)->load(std::memory_order_acquire);
  return TCPXU_SUCCESS;
}

int tcpxuEngineGetConfig(tcpxuEngine* e, tcpxuEngineConfig* config) {
  if (!e || !config) return TCPXU_INVALID_ARGUMENT;
  config->ring_entries = e->ring_entries;
  config->workgroups = e->workgroups;
  config->descs_per_ticket = e->per_ticket;
  config->spin_limit = e->spin_limit;
  return TCPXU_SUCCESS;
}

uint32_t tcpxuEngineCarriedDescs(void) { return kCarriedDescs; }

int tcpxuEngineDevice(tcpxuEngine* e, int* device) {
  if (!e || !device) return TCPXU_INVALID_ARGUMENT;
  *device = e->device;
  return TCPXU_SUCCESS;
}

int tcpxuEngineTicketPlan(uint32_t workgroups, uint32_t descs_per_ticket, uint32_t in_flight, uint32_t n_descs,
                          uint64_t payload_bytes, uint32_t* per_ticket, uint32_t* n_tickets, uint32_t* max_descs) {
  if (workgroups < 2 || workgroups > (1u << 16) || descs_per_ticket > kMaxDescsPerTicket || in_flight == 0) {
    set_error("ticket plan: 2..65536 workgroups, tickets of 0..%u, at least one submission in flight", kMaxDescsPerTicket);
    return TCPXU_INVALID_ARGUMENT;
  }
  const uint32_t limit = max_descs_for(descs_per_ticket);
  if (max_descs) *max_descs = limit;
  if (n_descs > limit) {
    set_error("%u descriptors in one submission exceed the limit of %u", n_descs, limit);
    return TCPXU_INVALID_ARGUMENT;
  }
  const uint32_t bytes = payload_bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : static_cast<uint32_t>(payload_bytes);
  const uint32_t per = descs_per_ticket != 0 ? descs_per_ticket
                                             : ticket_size_for_submission(in_flight, n_descs, bytes, workgroups - 1, false);
  if (per_ticket) *per_ticket = per;
  if (n_tickets) *n_tickets = (n_descs + per - 1) / per;
  return TCPXU_SUCCESS;
}

int tcpxuEngineRunning(tcpxuEngine* e, int* running) {
  if (!e || !running) return TCPXU_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(e->mu);
  *running = e->launched &&
             reinterpret_cast<std::atomic<uint64_t>*>(&e->ctl->exited)->load(std::memory_order_acquire) == 0;
  return TCPXU_SUCCESS;
}

}  // extern "C"
