// Device-side building blocks of the gfx950 unpack kernels: how one 64-lane wavefront moves fragments.
//
// A fragment is `len` bytes (at most one 4 KiB bounce page in practice) with arbitrary byte alignment on both
// sides.  The copy is organised around the DESTINATION: the body is written with aligned 16-byte vector stores
// that cover whole 128-byte lines wherever a neighbouring fragment continues the line, and byte-wise heads and
// tails remain only at the ends of a run of fragments.  Source vectors are fetched with 16-byte loads at the
// 4-byte aligned address just below where the destination alignment puts them and shifted into place in
// registers.  This is a pure bandwidth copy: no MFMA, no LDS for payload.
#ifndef TCPXU_UNPACK_DEVICE_H_
#define TCPXU_UNPACK_DEVICE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tcpx_unpack_hip.h"

namespace tcpxu {

constexpr int kWaveLanes = 64;
constexpr int kWgThreads = 256;
// Vectors a lane keeps in flight per round: 4 x 16 B x 64 lanes = one 4 KiB page per wavefront per round.
constexpr int kVecPerLane = 4;
constexpr uint32_t kVecPerRound = kVecPerLane * kWaveLanes;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Payload always lives in global memory (the arena and the caller's receive buffer), so every payload access
// is cast to the global address space: the compiler then emits global_* instead of flat_* instructions even
// where the address arrives as an integer.
#define TCPXU_GLOBAL __attribute__((address_space(1)))

// ---- the copy path ------------------------------------------------------------------------------------------------
// Scope of the payload accesses.  A kernel that never ends gets no cache invalidate at launch and no write-back
// at exit, so its payload accesses carry the coherence themselves: loads and stores are issued at system scope
// (sc0 sc1).  A load then never returns a line that an XCD's L2 kept from an earlier use of a recycled bounce
// page, and a store is written through, so that once the wavefront's memory counter has drained
// (s_waitcnt vmcnt(0)) the bytes are where the host, a DMA engine or another kernel will read them -- no L2
// write-back instruction is ever needed.  Plain launches use the same accesses: measured here they stream at
// least as fast as cached non-temporal ones.
typedef TCPXU_GLOBAL u32x4* gvec_ptr;
__device__ __forceinline__ u32x4 load_vec_sys(const uint8_t* p) {
  return __builtin_amdgcn_global_load_b128((gvec_ptr)p, "");
}
__device__ __forceinline__ void store_vec_sys(uint8_t* p, u32x4 v) {
  __builtin_amdgcn_global_store_b128((gvec_ptr)p, v, "");
}
// The bulk of the payload is stored with the non-temporal hint on top of the system scope (sc0 sc1 nt): the
// destination is written once and not read again by this kernel, and telling the caches so keeps it from
// displacing other data (at an 8 MiB chunk of 4 KiB fragments, all from HBM: 2.80 against 2.58 TB/s of payload).
// The hint on the loads as well measured no faster.  A round's stores go through windows (below), which take scope and hint
// as a number; the one here, for kernels that copy a single stretch, is written as an instruction, since no builtin
// combines the two on a plain address.  The s_nop covers the wait state the hardware wants between a store of more than
// 8 bytes and a write to its data registers, which the compiler cannot insert for an instruction it does not see.
__device__ __forceinline__ void store_vec_stream(uint8_t* p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" : : "v"((gvec_ptr)p), "v"(v) : "memory");
}
__device__ __forceinline__ uint32_t load_byte_sys(const uint8_t* p) {
  return __hip_atomic_load((const TCPXU_GLOBAL uint8_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void store_byte_sys(uint8_t* p, uint8_t v) {
  __hip_atomic_store((TCPXU_GLOBAL uint8_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Destination lines.  HBM with ECC punishes a 128-byte line that arrives as two partial writes, and with
// write-through stores no cache merges them.  Consecutive fragments of a message land back to back in the
// destination at arbitrary byte offsets, so almost every fragment boundary falls inside a line.  Rule: a line
// belongs to the fragment that holds its first byte.  The wavefront that copies fragment A also writes the rest
// of A's last line, taking those bytes from the source of the next fragment B, and the wavefront that copies B
// starts at B's first full line.  Every line inside a run of fragments is then written whole, by one wavefront.
// Both owners decide with the same inputs whether the rule applies to a boundary:
constexpr uint32_t kLineBytes = 128;
// The line must hold nothing but the end of A and the beginning of B -- A reaches back to the line's first byte, B
// on to its last -- and each of the two must be at least 16 bytes and not be one of the tiny fragments that are copied
// bytewise.
__device__ __forceinline__ bool fragment_is_tiny(const uint8_t* dst, uint32_t len);
__device__ __forceinline__ bool shares_line(uint64_t dst_a, uint32_t len_a, uint64_t dst_b, uint32_t len_b) {
  const uint32_t in_line = static_cast<uint32_t>(dst_a + len_a) & (kLineBytes - 1);  // bytes of A in the line
  return dst_a + len_a == dst_b && in_line != 0 && len_a >= in_line && len_a >= 16u && len_b >= kLineBytes - in_line &&
         len_b >= 16u && !fragment_is_tiny(reinterpret_cast<const uint8_t*>(dst_a), len_a) &&
         !fragment_is_tiny(reinterpret_cast<const uint8_t*>(dst_b), len_b);
}

// A window on memory: a buffer resource, whose accesses the hardware checks against its length, dword by dword.  A lane
// whose offset lies beyond it reads zeros without a trip to memory, and stores nothing: which lanes take part in an
// access costs no instruction.
typedef __amdgpu_buffer_rsrc_t Window;
__device__ __forceinline__ Window window(const uint8_t* p, uint32_t bytes) {
  constexpr int kRaw32 = 0x00020000;  // word 3: no swizzling, 32-bit data
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0, static_cast<int>(bytes), kRaw32);
}
constexpr uint32_t kOutside = 0x80000000u;       // an offset outside any window of a round's vectors or of a line
constexpr int kSystem = 17, kSystemStream = 19;  // scopes of a window's accesses: sc0 sc1; sc0 sc1 nt (see above)

// One round of a wavefront's copy work: up to 4 KiB of 16-byte vectors with a 16-byte aligned destination, the
// edge bytes of the fragment (a head and a tail of fewer than 16 bytes where the fragment keeps its own partial
// lines), and the shared last line (32 dwords, each from one of two sources, and one of them from both).
// Loading and storing are separate steps, with an explicit wait for everything in flight between them.
//
// Between them lie the instructions that bound rounds of short fragments (16 wavefronts a compute unit, each waiting for
// its own): so the vectors go through windows, with one offset per lane and no comparison, mask, branch or 64-bit address
// per vector, the line goes by dwords, where the boundary cuts one (by vectors, it took a shift by a number of dwords that
// the compiler made thirty branches of), and the edge bytes are not waited for ahead of the vectors.  A part of the round
// that has nothing to move is skipped by the whole wavefront.  (Against masked accesses and a line of eight vectors: 4 MiB
// of wire fragments in one launch 4.9 -> 4.4 us, 64 KiB of fragments of any length 4.2 -> 3.6, 256 MiB of them 99.6 -> 95.8,
// through the engine 113.7 -> 109.1; whole pages by the half GiB, which the memory system bounds, 0.3 % slower.)
constexpr uint32_t kNoEdge = 0xFFFFFFFFu;
struct CopyRound {
  // Wave-uniform (scalar registers):
  const uint8_t* src_vec;   // source of vector 0 of this round (any alignment)
  uint8_t* dst_vec;         // destination of vector 0 (16-byte aligned)
  const uint8_t* src_frag;  // first byte of the fragment
  uint8_t* dst_frag;
  const uint8_t* src_next;  // first byte of the next fragment's source if the last line is shared, else src_frag
  uint32_t nvec;            // vectors in this round, 0..kVecPerRound (0: nothing but a shared line or edge bytes)
  uint32_t frag_len;
  uint32_t line_off;        // offset of the shared last line from dst_frag
  uint32_t share_next;      // this round completes the fragment's last line out of the next fragment
  uint32_t edges;           // edge bytes that this round copies: head | tail << 8
};
constexpr int kDppWaveShiftLeft1 = 0x130;  // lane i receives lane i+1's value; lane 63 keeps the first operand
struct CopyRegs {
  u32x4 r[kVecPerLane];
  uint32_t line, line_next;  // the shared line's dwords from this fragment and from the next, zero where the other's are
  uint32_t tail_dword;       // the dword behind a round of kVecPerRound vectors, the same in every lane
  uint32_t edge_byte;
};

// The shared last line, lanes 0..31, a dword each.  The fragment (A) has `rem` = frag_len - line_off bytes in the line
// (1..127), the next fragment (B) the rest.  Dwords before the boundary are 4 bytes of A, dwords after it 4 bytes of B,
// loaded where they lie (any alignment) and stored as loaded.  The one dword that the boundary cuts (none if rem is a
// multiple of 4) is the last bytes of A followed by the first of B: its lane loads A's last 4 bytes, lane 32 loads B's first
// 4, and a shift of the two by the same amount for the whole wavefront makes it.  A load for each side, since a window has
// one base; a lane of the other side is outside and reads zero.  shares_line has seen to it that every one of these loads
// stays inside its fragment.
constexpr uint32_t kLineDwords = kLineBytes / 4;

// Source realignment.  A 16-byte load whose address is not a multiple of 4 is split by the memory pipeline and
// runs at roughly two thirds of the rate of one that is (a multiple of 4 that is not a multiple of 16 costs
// nothing).  Source and destination of a fragment are misaligned against each other by an arbitrary number of
// bytes, and the destination decides where vectors start, so the source address of a vector is arbitrary.  The
// round therefore loads from the 4-byte aligned address just below (`skew` = 0..3 bytes below, the same for
// every vector of the round) and shifts the bytes into place in registers: a vector is bytes [skew, skew+16)
// of its own four dwords plus one more dword, and that fifth dword is the first dword of the next vector --
// which the neighbouring lane holds.  For the round's last vector the window ends one dword further, so that the lane
// after it loads that dword and nothing else (with skew > 0 it starts inside the fragment, and an aligned dword never
// leaves the 4 KiB page it starts in; with skew 0 nothing of it is used and the window ends with the last vector).  A round
// of kVecPerRound vectors has no lane left for it and takes one load more.

// Lanes [0,head) carry the head, lanes [16,16+tail) the tail (both < 16 bytes); the other lanes have none.
__device__ __forceinline__ uint32_t edge_offset(const CopyRound& c, uint32_t lane) {
  const uint32_t in_tail = lane - 16u;
  uint32_t off = in_tail < (c.edges >> 8) ? c.line_off + in_tail : kNoEdge;
  if (lane < (c.edges & 0xFFu)) off = lane;
  return off;
}

__device__ __forceinline__ void round_load(const CopyRound& c, CopyRegs& x, uint32_t lane) {
  const uint32_t skew = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(c.src_vec)) & 3u;
  const uint8_t* base4 = c.src_vec - skew;
  const uint32_t at = lane << 4;
  // No register of the round is cleared first: what the shifts read from one that was not loaded never reaches a stored
  // byte.  The empty statement only tells the compiler that the registers have a value.
  asm volatile("" : "=v"(x.r[0]), "=v"(x.r[1]), "=v"(x.r[2]), "=v"(x.r[3]), "=v"(x.line), "=v"(x.line_next), "=v"(x.tail_dword),
               "=v"(x.edge_byte));
  if (c.share_next != 0) {  // (first: two source pages are asked for before the bulk of one of them)
    const uint32_t rem = c.frag_len - c.line_off, at4 = lane << 2;
    const bool in_next = at4 >= rem;
    const uint32_t own = in_next ? kOutside : min(at4 + 4u, rem);
    const uint32_t next = lane == kLineDwords ? 0u : in_next ? at4 - rem : kOutside;
    x.line = __builtin_amdgcn_raw_buffer_load_b32(window(c.src_frag + c.line_off - 4, rem + 4), own, 0, kSystem);
    x.line_next = __builtin_amdgcn_raw_buffer_load_b32(window(c.src_next, kLineBytes - rem > 4 ? kLineBytes - rem : 4), next, 0, kSystem);
  }
  const uint32_t bytes = ((c.nvec << 4) + skew + 3u) & ~3u;
  const Window from = window(base4, bytes);
#pragma unroll
  for (int k = 0; k < kVecPerLane; ++k) {
    constexpr uint32_t kStep = 16 * kWaveLanes;
    if (k == 0 || bytes > k * kStep) x.r[k] = __builtin_amdgcn_raw_buffer_load_b128(from, at + k * kStep, 0, kSystem);
  }
  if (bytes > 16 * kVecPerRound) x.tail_dword = __builtin_amdgcn_raw_buffer_load_b32(from, 16 * kVecPerRound, 0, kSystem);
  if (c.edges != 0)
    x.edge_byte = __builtin_amdgcn_raw_buffer_load_b8(window(c.src_frag, c.frag_len), edge_offset(c, lane), 0, kSystem);
}

// Waits for every load of the round (and for whatever else the wavefront has in flight) rather than let each
// vector be stored as soon as its own load has landed (what the compiler would arrange): the round's stores then
// leave back to back, which measured 2-3 % faster end to end.  The registers pass through the statement so that no
// use of them can be scheduled before it.
__device__ __forceinline__ void round_wait(CopyRegs& x) {
  asm volatile("s_waitcnt vmcnt(0)"
               : "+v"(x.r[0]), "+v"(x.r[1]), "+v"(x.r[2]), "+v"(x.r[3]), "+v"(x.line), "+v"(x.line_next),
                 "+v"(x.tail_dword), "+v"(x.edge_byte)
               :
               : "memory");
  static_assert(kVecPerLane == 4, "the statement above names the four vectors of a round");
}
// The same for two rounds whose loads are under way together.
__device__ __forceinline__ void rounds_wait(CopyRegs& x, CopyRegs& y) {
  round_wait(x);
  round_wait(y);
}

// Shifts the loaded bytes into place and stores them; the round's loads must have landed (round_wait).
__device__ __forceinline__ void round_store_loaded(const CopyRound& c, CopyRegs& x, uint32_t lane) {
  const uint32_t skew = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(c.src_vec)) & 3u;
  const uint32_t at = lane << 4;
  const uint32_t bytes = c.nvec << 4;
  const Window to = window(c.dst_vec, bytes);
#pragma unroll
  for (int k = 0; k < kVecPerLane; ++k) {
    constexpr uint32_t kStep = 16 * kWaveLanes;
    if (k != 0 && bytes <= k * kStep) continue;
    // First dword of the next vector: lane+1 of this register, or lane 0 of the next register for lane 63.
    // (a DPP wavefront shift, which leaves lane 63 what it is given: no trip through the LDS crossbar)
    const int wrap = k + 1 < kVecPerLane ? __builtin_amdgcn_readlane(static_cast<int>(x.r[k + 1 < kVecPerLane ? k + 1 : k][0]), 0)
                                         : static_cast<int>(x.tail_dword);
    const uint32_t next0 = static_cast<uint32_t>(
        __builtin_amdgcn_update_dpp(wrap, static_cast<int>(x.r[k][0]), kDppWaveShiftLeft1, 0xF, 0xF, false));
    u32x4 out;
    out[0] = __builtin_amdgcn_alignbyte(x.r[k][1], x.r[k][0], skew);
    out[1] = __builtin_amdgcn_alignbyte(x.r[k][2], x.r[k][1], skew);
    out[2] = __builtin_amdgcn_alignbyte(x.r[k][3], x.r[k][2], skew);
    out[3] = __builtin_amdgcn_alignbyte(next0, x.r[k][3], skew);
    __builtin_amdgcn_raw_buffer_store_b128(out, to, at + k * kStep, 0, kSystemStream);
  }
  if (c.share_next != 0) {
    const uint32_t rem = c.frag_len - c.line_off;
    x.line |= x.line_next;
    const uint32_t next4 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x.line), kLineDwords));
    const uint32_t cut = __builtin_amdgcn_alignbyte(next4, x.line, (0u - rem) & 3u);
    const uint32_t out = lane == rem >> 2 ? cut : x.line;
    __builtin_amdgcn_raw_buffer_store_b32(out, window(c.dst_frag + c.line_off, kLineBytes), lane << 2, 0, kSystemStream);
  }
  if (c.edges != 0)
    __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(x.edge_byte), window(c.dst_frag, c.frag_len), edge_offset(c, lane), 0, kSystem);
}

__device__ __forceinline__ void round_store(const CopyRound& c, CopyRegs& x, uint32_t lane) {
  round_wait(x);
  round_store_loaded(c, x, lane);
}

// A fragment too short to contain one destination-aligned vector (at most 30 bytes) is copied byte per lane,
// outside the round pipeline.
__device__ __forceinline__ bool fragment_is_tiny(const uint8_t* dst, uint32_t len) {
  const uint32_t head = static_cast<uint32_t>(-reinterpret_cast<uintptr_t>(dst)) & 15u;
  return len < head + 16u;
}
__device__ __forceinline__ void copy_tiny_fragment(const uint8_t* src, uint8_t* dst, uint32_t len, uint32_t lane) {
  if (lane < len) store_byte_sys(dst + lane, static_cast<uint8_t>(load_byte_sys(src + lane)));
}

// Where the vectors of a fragment that is not tiny start and end.
//   share_prev  the fragment's first partial line is written by the owner of the previous fragment
//   share_next  this owner completes the fragment's last line from src_next, the next fragment's source
struct FragmentPlan {
  uint32_t start_off;  // offset of vector 0 from the fragment's first byte
  uint32_t end_off;    // offset of the end of the last vector (where the shared last line starts, if there is one)
  uint32_t head, tail; // edge bytes before vector 0 and after the last vector, each fewer than 16
  uint32_t nvec;       // vectors in all; none where a short fragment lies in the shared lines of its two neighbours
};
__device__ __forceinline__ FragmentPlan plan_fragment(uint64_t dst_addr, uint32_t len, bool share_prev, bool share_next) {
  FragmentPlan p;
  p.head = 0;
  if (share_prev) {
    p.start_off = static_cast<uint32_t>(-dst_addr) & (kLineBytes - 1);
  } else {
    p.head = static_cast<uint32_t>(-dst_addr) & 15u;
    p.start_off = p.head;
  }
  p.tail = 0;
  if (share_next) {
    p.end_off = len - (static_cast<uint32_t>(dst_addr + len) & (kLineBytes - 1));
  } else {
    p.end_off = p.start_off + ((len - p.start_off) & ~15u);
    p.tail = len - p.end_off;
  }
  p.nvec = (p.end_off - p.start_off) >> 4;
  return p;
}
// The first round of a planned fragment; *nvec_left receives the vectors that remain for later rounds.
__device__ __forceinline__ CopyRound first_round_of(const uint8_t* src, uint8_t* dst, const uint8_t* src_next,
                                                    uint32_t len, bool share_next, uint32_t start_off,
                                                    uint32_t end_off, uint32_t head, uint32_t tail, uint32_t nvec,
                                                    uint32_t lane, uint32_t* nvec_left) {
  CopyRound c;
  c.src_frag = src;
  c.dst_frag = dst;
  c.src_vec = src + start_off;
  c.dst_vec = dst + start_off;
  c.src_next = share_next ? src_next : src;
  c.frag_len = len;
  c.line_off = end_off;
  c.share_next = share_next;
  c.edges = head | (tail << 8);
  c.nvec = nvec < kVecPerRound ? nvec : kVecPerRound;
  *nvec_left = nvec - c.nvec;
  return c;
}

// Copies descriptor i of a list of n with the calling wavefront (all arguments wave-uniform but `lane`): what the
// kernels that are launched per list do.  The descriptor before it, its own and the one after it are read into scalar
// registers: nothing is staged, nobody waits at a barrier.  They come through the scalar cache, which two compute units
// share and which is empty when a kernel begins (the list stays as it is until the kernel has ended, so that what it keeps
// is what is there): neighbouring wavefronts need the same lines, and with lists in the host's memory each request for one
// is a read over PCIe.  (By vector loads, two or three requests a wavefront -> so: 4 MiB of wire fragments, list in the
// host's memory, 4.20 -> 4.00 us, 1 MiB 3.53 -> 3.43; 512 MiB, list in the GPU's, 177.9 -> 176.7.  One load for a workgroup
// of 4, 8 or 16 wavefronts, handed over in LDS: 4 MiB 4.31, 4.31 and 4.97.)
// A fragment that is longer than a round takes several, the first with its edges and its shared line.
__device__ __forceinline__ void copy_descriptor(const uint8_t* bounce, uint8_t* dst, const tcpxuLoadMeta* descs, uint64_t n,
                                                uint64_t i, uint32_t lane) {
  typedef const __attribute__((address_space(4))) u32x4* constant_ptr;
  const constant_ptr list = (constant_ptr)(descs + i);
  const u32x4 none = {0u, 0u, 0u, 0u};
  const u32x4 d[3] = {i != 0 ? list[-1] : none, list[0], i + 1 < n ? list[1] : none};
  auto word = [&](int of, int k) { return d[of][k]; };
  auto place = [&](int of) { return reinterpret_cast<uint64_t>(dst) + ((static_cast<uint64_t>(word(of, 3)) << 32) | word(of, 2)); };
  constexpr int kPrev = 0, kOwn = 1, kNext = 2;
  const uint32_t len = word(kOwn, 1);
  if (len == 0) return;
  const uint64_t to = place(kOwn);
  const uint8_t* from = bounce + word(kOwn, 0);
  uint8_t* const to_ptr = reinterpret_cast<uint8_t*>(to);
  if (fragment_is_tiny(to_ptr, len)) {
    copy_tiny_fragment(from, to_ptr, len, lane);
    return;
  }
  // (Past either end of the list the neighbour reads as empty, and an empty fragment shares nothing.)
  const bool share_prev = shares_line(place(kPrev), word(kPrev, 1), to, len);
  const bool share_next = shares_line(to, len, place(kNext), word(kNext, 1));
  const FragmentPlan p = plan_fragment(to, len, share_prev, share_next);
  uint32_t left;
  CopyRound r = first_round_of(from, to_ptr, share_next ? bounce + word(kNext, 0) : from, len, share_next, p.start_off, p.end_off,
                               p.head, p.tail, p.nvec, lane, &left);
  CopyRegs x;
  for (;;) {
    round_load(r, x, lane);
    round_store(r, x, lane);
    if (left == 0) return;
    r.edges = 0;
    r.share_next = 0;
    r.src_vec += static_cast<size_t>(r.nvec) << 4;
    r.dst_vec += static_cast<size_t>(r.nvec) << 4;
    r.nvec = left < kVecPerRound ? left : kVecPerRound;
    left -= r.nvec;
  }
}

// The 8 XCDs of an MI355X receive workgroups round-robin by workgroup id and each has its own L2.  This maps a
// workgroup id to a work-item index such that neighbouring items meet on one XCD: they have a destination line and the
// lines that their descriptors come in in common.
//
// In a short list every XCD takes one contiguous eighth: its descriptors arrive a line at a time, over PCIe perhaps.  In a
// longer one it takes runs of kXcdRunDescs in turn, so that what is being written at a time is one stretch of the destination
// and not eight of them, each an eighth of the message away from the next.  (Groups of four descriptors, contiguous eighths
// / runs of 1 / 8 / 24 / 32 / 64, us: 512 MiB of wire fragments 177.3 / 172.8 / 172.0 / 172.3 / 174.5 / 174.1, of whole pages
// 194.3 / 191.0 / 191.1 / 190.7 / 189.7 / 189.5, 256 MiB of whole pages 98.0 / 95.7 / 96.6 / 95.7 / 95.4 / 95.9, of ragged
// fragments 94.6 / 90.9 / 90.9 / 90.8 / 90.7 / 91.3, 64 MiB of wire fragments 25.3 / 24.2 / 24.2 / - / 24.3 / -; runs of 4 and 12 are
// worse for whole pages, 203.8 and 198.6.  A slot of 4 MiB whose list is in the host's memory 3.95 / 4.53 / 4.02 / - / 4.04 / -;
// 8 MiB, 2155 descriptors, 4.75 and 4.79 in runs of 24, 16 MiB 8.67 and 8.65.)
constexpr uint32_t kXcds = 8;
constexpr uint32_t kXcdRunDescs = 96;
__device__ __forceinline__ uint32_t xcd_near_index(uint32_t wg, uint32_t items, uint32_t contiguous_up_to, uint32_t run) {
  if (items <= contiguous_up_to) {
    const uint32_t per_xcd = (items + kXcds - 1) / kXcds;
    return (wg % kXcds) * per_xcd + wg / kXcds;  // may be >= items: caller skips
  }
  const uint32_t turn = wg / (kXcds * run) * (kXcds * run);  // the first item of this turn, and its first workgroup
  if (turn + kXcds * run > items) return wg;                 // (what is left beyond whole turns; caller skips as above)
  return turn + (wg % kXcds) * run + (wg - turn) / kXcds;
}

}  // namespace tcpxu

#endif  // TCPXU_UNPACK_DEVICE_H_
