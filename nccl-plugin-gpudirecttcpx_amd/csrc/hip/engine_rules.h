// What the engine decides by numbers alone.  No device code and no HIP header: tests compile it on the host.
#ifndef TCPXU_ENGINE_RULES_H_
#define TCPXU_ENGINE_RULES_H_

#include <stdint.h>

// (The leader works out ticket sizes on the GPU with what the host works out for tcpxuEngineTicketPlan and bursts.)
#if defined(__HIP__)
#define TCPXU_RULE __host__ __device__ __forceinline__
#else
#define TCPXU_RULE inline
#endif

namespace tcpxu {
namespace {

constexpr uint32_t kMaxDescsPerTicket = 64;
// Ticket size when the caller does not fix one.  A ticket occupies a workgroup for one pick-up (a claim, the
// ticket record, the descriptors over PCIe: a few microseconds) plus its copy.  While workgroups are waiting for
// work, small tickets finish a submission sooner (more workgroups share it); once tickets queue up behind busy
// workgroups, larger ones spend less of each workgroup's time on pick-ups.  `backlog` estimates the descriptors of
// all submissions not yet completed, counting each in full until it completes (how far the slots in flight have
// got depends on the ticket size itself and would feed back).  The steps are where throughput measured at 1 to
// 64 slots of 4 MiB in flight changed hands between sizes; 8 is one fragment per copy wavefront, 16 two.  Beyond
// 16 nothing is gained for fragments of a page: with every source page coming from HBM, 64 slots in flight move
// 71.0 % of the roofline in tickets of 16, 70.1 % in tickets of 24 and 69.4 % in tickets of 32 (more tickets than
// workgroups keep every workgroup supplied, and a wavefront that has finished its share waits less for the
// slowest one).
// (Descriptors per worker workgroup below 13, 18; written without the division, which the leader would pay for
// on every submission.  backlog <= 2^20 and workers < 2^16 keep the products in 32 bits.)
TCPXU_RULE uint32_t ticket_size_for(uint32_t backlog, uint32_t workers) {
  return backlog < 13u * workers ? 8u : backlog < 18u * workers ? 12u : 16u;
}
// ceil(n / per_ticket) for 1 <= n <= 2^20 and 1 <= per_ticket <= 64 without the forty-odd instructions of a general
// 32-bit division: the quotient estimated in floating point (both operands are exact there) and put right by at most one.
TCPXU_RULE uint32_t tickets_for(uint32_t n, uint32_t per_ticket) {
  const uint32_t x = n + per_ticket - 1;
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t q = static_cast<uint32_t>(static_cast<float>(x) * __builtin_amdgcn_rcpf(static_cast<float>(per_ticket)));
#else
  uint32_t q = static_cast<uint32_t>(static_cast<float>(x) / static_cast<float>(per_ticket));
#endif
  while (q * per_ticket > x) --q;
  while (x - q * per_ticket >= per_ticket) ++q;
  return q;
}
// Ticket size for one submission of n descriptors when `in_flight` submissions (this one included) are not yet
// completed; each is taken to be as long as this one.  A small submission among many stays whole: with 8 or
// more in flight the parallelism is in the submissions, and a submission that is one ticket costs the leader
// one store instead of a pass of its loop.  (64 KiB requests of 16 fragments, p50 publish -> done: 8.7 -> 9.1 us
// at 8 in flight, 17.5 -> 9.3 us at 32, where the leader's loop had become the queue.)
//
// `bytes` is the submission's payload if the caller said (0 = unknown: whole pages).  The largest step, 16, stands
// for whole pages (14 while the backlog is shallow, see below: seven copy wavefronts then get two fragments each and
// one gets none); a submission of shorter fragments gets more descriptors per ticket, in multiples of 16 so that
// the copy wavefronts' shares come out even, up to 64 (full_ticket_size).  Written as comparisons: the leader runs
// this for every submission and a division costs it forty instructions.
constexpr uint32_t kManyInFlight = 8, kSmallSubmission = 32;
constexpr uint32_t kCarriedDescs = 16;  // descriptors that travel with a submission, and then with its one ticket (see CarriedList)
constexpr uint32_t kLaneTickets = 32;  // tickets of one submission that the lanes holding its entry still write themselves
// Entries waiting in one poll from which the leader counts as the bottleneck and makes no tickets of fewer than 16: eight,
// or four for entries whose backlog asks for fewer than 14.  A look comes round twice as often as a poll that asks when the
// last is done, and shows half as many.  (Four requests of 4 MiB in one call, 8.7 descriptors a workgroup: 20.8 us with 8
// throughout, where the tickets of 8 that the backlog asks for are a few more than there are workgroups, 16.8 with 4 or 3;
// 64 of 1 MiB 29.0 and 28.8, streams of 1 MiB requests and storms the same.  Tickets of 14 are a stream's, which four
// entries in one look say nothing about: one comm's sixteen slots 70.9 % of the roofline with 4 throughout, 71.8 with 8 for
// those; raised to 14 only, five requests of 4 MiB take 18.2 us instead of 17.3.)
constexpr uint32_t kLeaderBehind = 8, kLeaderBehindShallow = 4;
constexpr uint32_t kFullTicket = 16, kStreamTicket = 14;
constexpr uint32_t kDeepBacklog = 100;  // descriptors per worker workgroup from which whole pages go in tickets of 16
TCPXU_RULE uint32_t full_ticket_size(uint32_t bytes, uint32_t n) {
  static_assert(kFullTicket == 16 && kMaxDescsPerTicket == 64, "the steps below");
  const uint64_t b = bytes;  // n <= 2^20: the products need more than 32 bits
  // Whole pages (or no hint): 16.  Shorter fragments: 32 from two thirds of a page down, 48 from half a page down,
  // 64 below a third -- about 96 KiB a ticket rather than 64, because a round of a short fragment costs a wavefront
  // nearly what a whole page costs and only a larger share per pick-up makes up for it (fragments of 1.8 KiB on
  // average, 64 slots in flight: 59.6 % of the roofline in tickets of 32, 60.6 % in 40, 61.1 % in 48, 61.3 % in 64).
  return bytes == 0 || b >= 2731ull * n ? 16u : b >= 2048ull * n ? 32u : b >= 1366ull * n ? 48u : 64u;
}
// Ticket size for a call's submissions of whole pages where it hands over kManyInFlight or more, between 12 and 40
// descriptors per worker workgroup in all.  A burst does not go on as a stream does: by backlog, its submissions are cut as
// small as what the leader has seen of it so far asks for, and the last round is nearly empty.  Microseconds a call, with
// other buffers from pass to pass, by backlog / in tickets of 18 / 20 / 22 / 24: eight requests of 4 MiB 24.9 / 24.2 / 24.4 /
// 25.1 / 25.4, sixteen 35.5 / 35.6 / 36.1 / 36.5 / 36.6, 16 of 2 MiB 26.1 / 24.3 / 24.2 / 24.2 / 24.3, 32 of 2 MiB 38.5 / 36.1 /
// 36.6 / 36.9 / 37.0, 40 of 1 MiB 28.9 / 28.9 / 29.7 / 29.9 / 29.9, 64 of 1 MiB 35.8 / 35.7 / 35.8 / 36.1 / 35.5.  Where a part of
// the buffers is still in the caches, sixteen of 4 MiB take 33.5 by backlog and 32.6 with 18 to 24 (on some machines 31.8 and
// 32.5).  Above the range the last round is a small part of the whole (24 requests of 4 MiB, 48 a workgroup: 46.5 by backlog,
// 47.3 in tickets of 18); below it the sizes by backlog, which begin at 8, reach all the workgroups sooner.
constexpr uint32_t kBurstTicket = 18;
// Ticket size for submissions of fragments of a third to half a page (the step of 48) where a call hands over kManyInFlight or
// more, or while the backlog is shallow: 32.  What is being written at a time is then a narrower stretch of the destination,
// which the memory takes faster, and the last round is shorter.  (48 / 32, us a call of fragments of 850 to 2550 or 925 to 2775
// bytes, requests of so many of them: 16 of 1000 23.2 / 22.6, 64 of 1000 53.4 / 52.8, 8 of 1600 21.0 / 19.1, 16 of 1600 26.8 /
// 25.9, 64 of 1600 77.6 / 75.8, 86 of 1700 110.2 / 107.8.  A stream of 1 MiB requests, 64 in flight, 4.86 / 5.22 TB/s r+w.)
// Not for:
// * Requests of 1025 to 1536 fragments, of which the leader writes tickets of 48 from the entry's lanes and tickets of 32 one
//   entry after the other.  That costs it up to a microsecond a request, which is what requests of up to 2.2 MB are copied in:
//   in calls of 64, of 1030 fragments 55.7 us / 65.8, 1200 62.5 / 67.0, 1400 of 1500 bytes 65.5 / 67.0, but 1400 of 1700 bytes
//   71.8 / 69.9 and 1530 77.5 / 73.8; calls of 8 and 16 are 3 to 10 % faster in tickets of 32 from 1200 on.  Streams of 1280,
//   in flight 8 / 16 / 32 / 64: 2.09 / 3.19 / 4.59 / 5.31 TB/s in tickets of 48, 2.48 / 3.71 / 4.57 / 4.50 in tickets of 32 while
//   shallow.  The line is where nothing loses.
// * Calls of kLongBurst descriptors per worker and more, whose last round is nothing beside the rest: 250 of 1000 fragments
//   162.9 us / 163.2, 512 310.3 / 312.9, 1000 584.5 / 592.3 (300 of 1700, below the line, 329.8 / 328.8).
// * Calls that find kAheadOfBurst descriptors per worker queued already: a stream, which larger tickets move faster once it
//   is deep, and which has no last round.  Calls of 16 requests, other calls under way 1 / 2 / 3 / 7, TB/s r+w: of 1700 fragments
//   6.30 / 7.27 / 6.20 / 5.96 in tickets of 48, 6.55 / 7.16 / 6.08 / 5.94 in tickets of 32, 6.79 / 7.05 / 6.22 / 5.96 by this line;
//   of 1000 fragments, 1 / 3 / 7, 4.36 / 6.98 / 5.56 in tickets of 48, 4.15 / 6.94 / 5.46 in tickets of 32, 4.15 / 6.80 / 5.56 by this line.
//   (With two and three calls in the caches it is the leader that a stream waits for, and working out a size by backlog takes it
//   longer than reading the mark.)
// * Streams of more than 1024 fragments a request, whose leader would have that microsecond to spend on each.
constexpr uint32_t kShortBurstTicket = 32, kShortTicket = 48;
constexpr uint32_t kLongBurst = 1000, kAheadOfBurst = 40;
inline bool burst_of_short_fragments(uint32_t submissions, uint32_t n, uint32_t bytes, uint32_t workers) {
  const uint64_t all = static_cast<uint64_t>(submissions) * n;
  return submissions >= kManyInFlight && n > kSmallSubmission && full_ticket_size(bytes, n) == kShortTicket &&
         all >= 18ull * workers && all < 1ull * kLongBurst * workers;
}
inline bool few_ahead_of_burst(uint64_t submissions_ahead, uint32_t n, uint32_t workers) {
  return submissions_ahead * n < 1ull * kAheadOfBurst * workers;
}
inline bool burst_of_pages(uint32_t submissions, uint32_t n, uint32_t bytes, uint32_t workers) {
  const uint64_t all = static_cast<uint64_t>(submissions) * n;
  return submissions >= kManyInFlight && n > kSmallSubmission && full_ticket_size(bytes, n) == kFullTicket &&
         all >= 12ull * workers && all < 40ull * workers;
}
TCPXU_RULE uint32_t ticket_size_for_submission(uint32_t in_flight, uint32_t n, uint32_t bytes, uint32_t workers, bool burst) {
  if (burst) {
    const uint32_t full = full_ticket_size(bytes, n);
    const bool same_way = n <= kLaneTickets * kShortBurstTicket || n > kLaneTickets * kShortTicket;
    return full == kFullTicket ? kBurstTicket : full == kShortTicket && same_way ? kShortBurstTicket : full;
  }
  if (n <= kCarriedDescs) return kCarriedDescs;
  if (in_flight >= kManyInFlight && n <= kSmallSubmission) return kSmallSubmission;
  const uint64_t all = static_cast<uint64_t>(in_flight) * n;
  const uint32_t backlog = all > (1u << 20) ? (1u << 20) : static_cast<uint32_t>(all);
  const uint32_t size = ticket_size_for(backlog, workers);
  if (size < kFullTicket) return size;
  const uint32_t full = full_ticket_size(bytes, n);
  if (full > kFullTicket)
    return full == kShortTicket && n <= kLaneTickets * kShortBurstTicket && backlog < kDeepBacklog * workers ? kShortBurstTicket : full;
  // Whole pages and a backlog that is there but not deep (one comm's sixteen slots of 4 MiB are 34 descriptors per
  // workgroup: every workgroup holds a ticket and has the next one staged, and hardly any wait unclaimed): tickets
  // of 14 make a seventh more of them, and the workgroups run dry less often -- one comm 71.1 -> 72.2 % of the
  // roofline, two to four comms the same as with 16 (72.4-72.5 %).
  return backlog < kDeepBacklog * workers ? kStreamTicket : kFullTicket;
}

// Room in the ticket ring.  `out` and `known_done` are low words of running counts: of the tickets written, and of those that the
// leader knows to be done, which may be fewer than are (it does not read that count with every look, see leader_loop).
constexpr uint32_t kTicketRing = 1u << 16;  // tickets in flight at most
// (None, and not four billion, where the two say that more are out than the ring holds.  A signed maximum is one scalar
// instruction; a comparison of the two counts becomes a vector subtraction and a trip back, in every look that shows an entry.)
TCPXU_RULE uint32_t ticket_room(uint32_t out, uint32_t known_done) {
  const int32_t room = static_cast<int32_t>(kTicketRing - (out - known_done));
  return room > 0 ? static_cast<uint32_t>(room) : 0u;
}
// Whether to ask how many are done: whenever an entry that is there could not be handed out, however few tickets are out (one
// entry's may need the whole ring, and nothing else would ever tell the leader that the ring has emptied), and before that
// once the ring may be half full, so that streams hardly ever come to wait.
TCPXU_RULE bool ask_what_is_done(uint32_t out, uint32_t known_done, bool entry_waits) {
  return entry_waits || out - known_done > kTicketRing / 2;
}
// What is known once the count has been read.  It can say less than is known already: a workgroup counts a ticket and, where that
// is the submission's last, the submission with two additions to different lines and waits for neither, so that the leader can
// see all submissions completed, and take all tickets for done, before the last tickets are counted.  They are done all the same.
// (Far less than half the range is written between two readings: a difference of that or more is a step back.)
TCPXU_RULE uint32_t known_done_after(uint32_t known_done, uint32_t counted) {
  return static_cast<int32_t>(counted - known_done) > 0 ? counted : known_done;
}

// The leader has its compute unit to itself.  Loads seem to return to a compute unit in the order in which it issued them,
// so the looks at the host's ring and the copy's loads wait for each other where both are under way.  A worker workgroup
// that finds itself there claims no ticket and leaves (its place then goes to the one workgroup of the grid that found
// none, which does the same) -- provided that this many others have started elsewhere: one that is placed while other
// kernels hold most of the GPU keeps all of its workers.  (Requests of 64 KiB: 2048 in one call 67.5 -> 63.5 us,
// 1024 41.4 -> 39.3, 16 to 256 within 2 % either way; a stream with 1024 in flight 40.5 -> 48.5 M/s, one comm's sixteen slots
// of 4 MiB 71.9 -> 72.5 % of the roofline; large requests the same, so two workers of 512 are not missed.)
constexpr uint32_t kEnoughElsewhere = 256;
// Whether a grid of so many workgroups can come to that many, with the leader and one worker on the leader's compute unit.  In
// a smaller one the leader says that it is nowhere, so that no worker waits for others to start or asks for them later.  (Said by
// the leader, once: asked by the workers, calls of 16 requests of 64 KiB take 10.45 us instead of 10.05, since the compiler
// then makes something else of the fetcher's loop.)
constexpr bool enough_can_be_elsewhere(uint32_t workgroups) { return workgroups >= kEnoughElsewhere + 2; }

}  // namespace
}  // namespace tcpxu
#endif  // TCPXU_ENGINE_RULES_H_
