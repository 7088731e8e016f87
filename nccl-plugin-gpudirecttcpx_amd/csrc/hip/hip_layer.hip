// HIP layer of the receive-side unpack path: device selection, the bounce-page arena, mapped queue memory and
// the launch-per-batch unpack kernel, all behind the C-ABI of include/tcpx_unpack_hip.h.
// The persistent engine lives in engine.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "hip_common.h"
#include "tcpx_unpack_hip.h"
#include "unpack_device.h"

namespace tcpxu {

thread_local char g_last_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof g_last_error, fmt, ap);
  va_end(ap);
}

namespace {

// Launch-per-batch unpack: one wavefront per descriptor, in workgroups of kWaves, as many workgroups as it takes.
//
// What bounds a short list is the chain launch -> descriptor -> payload -> store, each link a trip to memory; what
// bounds a long one is the memory system, and for short fragments how many wavefronts keep loads in flight.  Hence no
// LDS, no barrier and nothing carried from one fragment to the next: the descriptors go from the load into scalar
// registers, every wavefront of the 32 that a compute unit holds has a fragment of its own, and the dispatcher hands
// out new ones as they finish.  (Against workgroups of twelve wavefronts that staged their batch's descriptors in LDS,
// where a list of up to 8192 kept four of the twelve busy: 16 fragments 2.9 -> 2.4 us a launch (what the host needs for
// one), 4 MiB of wire fragments 5.1 -> 4.3 us, 8 MiB 6.6 -> 5.0, 16 MiB 10.0 -> 7.0, 64 MiB 23.6 -> 22.4; 256 MiB of
// 1.8 KiB fragments 126-140 -> 99 us; since then, with the round of unpack_device.h, descriptors by scalar loads and XCDs in
// turn: 4 MiB 3.8, 64 MiB 24.2, 256 MiB of 1.8 KiB fragments 90.8 = 5.9 TB/s r+w.  Those want all 32 wavefronts -- with 24 / 16
// resident 98.7 / 116.5 us where 32 took 95.5 -- while long fragments want fewer, 512 MiB of wire fragments 176.2 / 172.9 where
// 32 took 178.3, and the list does not say which they are.  Two descriptors per wavefront with 16 resident: 180.4 and 102.
// Half a fragment per wavefront, or two wavefronts to a workgroup, measured no better for short lists.)
//
// A wavefront is a workgroup of its own in lists of up to kShortList descriptors: nobody waits for three others to be placed
// or to finish.  In longer ones four begin together, and what is written at a time is a little more compact.  (Workgroups of
// one / two / four wavefronts, us a launch with other buffers from pass to pass: 4 MiB of wire fragments, list in the host's
// memory, 3.53 / 3.60 / 3.79, 3 MiB of ragged ones 4.07 / 4.09 / 4.15; list in the GPU's memory, 8 MiB of wire fragments 3.42 /
// 3.45 / 3.52, 16 MiB 6.26 / 6.29 / 6.38, 16 MiB of ragged ones, 9100 descriptors, 7.35 / 7.34 / 7.30, 256 MiB of them 92.9 / 92.4 /
// 92.5, 512 MiB of wire fragments 170.4 / 170.8 / 171.1, of whole pages 191.3 / 191.6 / 191.4.  Of eight and sixteen, 4 MiB 3.70
// and 4.45.)
constexpr uint64_t kShortList = 8192;
constexpr uint32_t kLongListWaves = 4;
constexpr uint32_t kContiguousDescs = 4096;  // see xcd_near_index
template <uint32_t kWaves>
__global__ __launch_bounds__(kWaves* kWaveLanes) __attribute__((amdgpu_waves_per_eu(8))) void unpack_batch_kernel(
    const uint8_t* __restrict__ bounce, uint8_t* __restrict__ dst, const tcpxuLoadMeta* __restrict__ descs,
    uint64_t n_descs, uint64_t first_group, uint32_t n_groups) {
  static_assert(kXcdRunDescs % kWaves == 0 && kContiguousDescs % kWaves == 0, "whole workgroups");
  const uint32_t lane = threadIdx.x & (kWaveLanes - 1);
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWaveLanes)));
  const uint32_t group = xcd_near_index(blockIdx.x, n_groups, kContiguousDescs / kWaves, kXcdRunDescs / kWaves);
  if (group >= n_groups) return;
  const uint64_t i = (first_group + group) * kWaves + wave;
  if (i < n_descs) copy_descriptor(bounce, dst, descs, n_descs, i, lane);
}

// One slot with a completion word (tcpxuUnpackSlotNoAlloc).  The word may be written once every wavefront's stores are
// acknowledged, and nothing that a kernel could count that in is its own: a fixed array of counters is shared by whatever
// runs at the same time (two executables of one captured graph pass the same arguments), and then the word comes early or
// never.  So up to kSmallSlot descriptors are one workgroup, which knows by its barrier, and a longer list is the kernel
// above followed by one of one thread that writes the word: the order of the stream says the rest.  A workgroup has sixteen
// wavefronts at the most, so beyond 16 descriptors some of them take two, one after the other, while a second launch costs
// the host 2.8 us.  (Us a call, one workgroup / two launches: 18 whole pages 4.2 / 6.3, 20 4.35 / 6.3, 24 4.9 / 6.3, 32 5.9 / 6.3,
// 40 7.1 / 6.3; a call that is waited for: 24 pages 15.4 / 15.9, 32 16.6 / 15.8.)
//
// The line lies where it does for fragments of up to a page.  What one workgroup does not do well is bytes, 128 KiB in and out
// of one compute unit for 3 us; of longer fragments it takes fewer to reach that (24 of 4 KiB 5.0 / 5.9, of 6 KiB 6.4 / 5.9, of 64 KiB
// 35.7 / 11.0; 17 of 6 KiB 5.2 / 5.9, of 9000 bytes 6.7 / 6.0; 16 of 8 KiB 5.5 / 5.9, of 16 KiB 8.2 / 5.9; 8 of 16 KiB 5.3 / 6.0, of
// 64 KiB 12.9 / 11.0; 4 of 64 KiB 11.0 / 10.9).  The host does not know the lengths -- a call may be captured or queued before
// its list is written -- so the entry point's description says what that costs and how a caller of such lists avoids it.
constexpr uint32_t kSmallSlot = 24;
constexpr uint32_t kSmallSlotWaves = 16;
__global__ __launch_bounds__(kSmallSlotWaves* kWaveLanes) void unpack_small_slot_kernel(const uint8_t* __restrict__ bounce, uint8_t* __restrict__ dst,
                                                                                  const tcpxuLoadMeta* __restrict__ descs, uint32_t n_descs,
                                                                                  uint64_t* done_flag, uint64_t done_value) {
  const uint32_t lane = threadIdx.x & (kWaveLanes - 1);
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWaveLanes)));
  for (uint32_t i = wave; i < n_descs; i += kSmallSlotWaves) copy_descriptor(bounce, dst, descs, n_descs, i, lane);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this wavefront's write-through stores are acknowledged
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(done_flag, done_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// The word of a longer slot, in stream order after its bytes, or of an empty one.
__global__ void complete_slot_kernel(uint64_t* done_flag, uint64_t done_value) {
  __hip_atomic_store(done_flag, done_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct DeviceProps {
  std::atomic<bool> valid{false};
  int compute_units = 0;
  char name[256] = "";
};
DeviceProps g_props[kMaxDevices];

}  // namespace

bool device_known(int device) { return device >= 0 && device < kMaxDevices && g_props[device].valid.load(std::memory_order_acquire); }

int use_device(int device) {
  if (device < 0 || device >= kMaxDevices) {
    set_error("device index %d out of range", device);
    return TCPXU_INVALID_ARGUMENT;
  }
  TCPXU_HIP(hipSetDevice(device));
  if (!device_known(device)) {
    hipDeviceProp_t p;
    TCPXU_HIP(hipGetDeviceProperties(&p, device));
    g_props[device].compute_units = p.multiProcessorCount;
    snprintf(g_props[device].name, sizeof g_props[device].name, "%s (%s)", p.name, p.gcnArchName);
    g_props[device].valid.store(true, std::memory_order_release);
  }
  return TCPXU_SUCCESS;
}

int device_compute_units(int device) { return g_props[device].compute_units; }

namespace {
std::mutex g_mapped_mu;
std::vector<MappedView::Block> g_mapped;  // by device address
std::atomic<uint64_t> g_mapped_generation{1};

void mapped_block_added(void* host, void* dev, size_t bytes) {
  std::lock_guard<std::mutex> lock(g_mapped_mu);
  const MappedView::Block b{reinterpret_cast<uintptr_t>(dev), reinterpret_cast<uintptr_t>(host), bytes};
  g_mapped.insert(std::upper_bound(g_mapped.begin(), g_mapped.end(), b, [](const auto& x, const auto& y) { return x.dev < y.dev; }), b);
  g_mapped_generation.fetch_add(1, std::memory_order_release);
}
void mapped_block_removed(void* host) {
  std::lock_guard<std::mutex> lock(g_mapped_mu);
  const uintptr_t h = reinterpret_cast<uintptr_t>(host);
  g_mapped.erase(std::remove_if(g_mapped.begin(), g_mapped.end(), [h](const auto& b) { return b.host == h; }), g_mapped.end());
  g_mapped_generation.fetch_add(1, std::memory_order_release);
}
}  // namespace

const void* mapped_host_address(MappedView* view, const void* dev, size_t bytes) {
  if (view->generation != g_mapped_generation.load(std::memory_order_acquire)) {
    std::lock_guard<std::mutex> lock(g_mapped_mu);
    view->blocks = g_mapped;
    view->generation = g_mapped_generation.load(std::memory_order_relaxed);
  }
  const uintptr_t at = reinterpret_cast<uintptr_t>(dev);
  auto b = std::upper_bound(view->blocks.begin(), view->blocks.end(), at, [](uintptr_t a, const auto& x) { return a < x.dev; });
  if (b == view->blocks.begin()) return nullptr;
  --b;
  if (bytes > b->bytes || at - b->dev > b->bytes - bytes) return nullptr;
  return reinterpret_cast<const void*>(b->host + (at - b->dev));
}

}  // namespace tcpxu

using namespace tcpxu;

extern "C" {

const char* tcpxuLastError(void) { return g_last_error; }

int tcpxuDeviceCount(int* count) {
  if (!count) return TCPXU_INVALID_ARGUMENT;
  *count = 0;
  TCPXU_HIP(hipGetDeviceCount(count));
  return TCPXU_SUCCESS;
}

int tcpxuDeviceInfo(int device, char* name, size_t name_len, int* compute_units) {
  TCPXU_TRY(use_device(device));
  if (name && name_len) snprintf(name, name_len, "%s", g_props[device].name);
  if (compute_units) *compute_units = g_props[device].compute_units;
  return TCPXU_SUCCESS;
}

int tcpxuArenaCreate(int device, size_t bytes, void** arena_base) {
  if (!arena_base || bytes == 0 || bytes % TCPXU_PAGE_SIZE != 0) {
    set_error("arena size %zu must be a positive multiple of %d", bytes, TCPXU_PAGE_SIZE);
    return TCPXU_INVALID_ARGUMENT;
  }
  if (bytes > (1ull << 32)) {
    set_error("arena size %zu exceeds the 4 GiB reach of a 32-bit src_off", bytes);
    return TCPXU_INVALID_ARGUMENT;
  }
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipMalloc(arena_base, bytes));
  if (reinterpret_cast<uintptr_t>(*arena_base) % TCPXU_PAGE_SIZE != 0) {
    (void)hipFree(*arena_base);
    *arena_base = nullptr;
    set_error("arena base is not page aligned");
    return TCPXU_INTERNAL_ERROR;
  }
  return TCPXU_SUCCESS;
}

int tcpxuArenaDestroy(int device, void* arena_base) {
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipFree(arena_base));
  return TCPXU_SUCCESS;
}

int tcpxuDeviceAlloc(int device, size_t bytes, void** ptr) {
  if (!ptr || bytes == 0) return TCPXU_INVALID_ARGUMENT;
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipMalloc(ptr, bytes));
  return TCPXU_SUCCESS;
}

int tcpxuDeviceFree(int device, void* ptr) {
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipFree(ptr));
  return TCPXU_SUCCESS;
}

int tcpxuCopyToDevice(int device, void* dst_dev, const void* src_host, size_t bytes) {
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipMemcpy(dst_dev, src_host, bytes, hipMemcpyHostToDevice));
  return TCPXU_SUCCESS;
}

int tcpxuCopyToHost(int device, void* dst_host, const void* src_dev, size_t bytes) {
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipMemcpy(dst_host, src_dev, bytes, hipMemcpyDeviceToHost));
  return TCPXU_SUCCESS;
}

int tcpxuFillDevice(int device, void* dst_dev, int byte_value, size_t bytes) {
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipMemset(dst_dev, byte_value, bytes));
  TCPXU_HIP(hipDeviceSynchronize());
  return TCPXU_SUCCESS;
}

int tcpxuDeviceSynchronize(int device) {
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipDeviceSynchronize());
  return TCPXU_SUCCESS;
}

int tcpxuMappedAlloc(int device, size_t bytes, void** host_ptr, void** dev_ptr) {
  if (!host_ptr || !dev_ptr || bytes == 0) return TCPXU_INVALID_ARGUMENT;
  TCPXU_TRY(use_device(device));
  TCPXU_HIP(hipHostMalloc(host_ptr, bytes, hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable));
  memset(*host_ptr, 0, bytes);
  TCPXU_HIP(hipHostGetDevicePointer(dev_ptr, *host_ptr, 0));
  mapped_block_added(*host_ptr, *dev_ptr, bytes);
  return TCPXU_SUCCESS;
}

int tcpxuMappedFree(int device, void* host_ptr) {
  TCPXU_TRY(use_device(device));
  mapped_block_removed(host_ptr);
  TCPXU_HIP(hipHostFree(host_ptr));
  return TCPXU_SUCCESS;
}

// ---- device memory that the host can write ------------------------------------------------------------------------
// Fine-grained device memory is mapped for the host through the PCIe BAR where the whole of device memory is
// exposed (large BAR).  Blocks are small and few, and they are handed back to a pool, never to the driver:
// memory with non-default caching is not returned while the process lives.
namespace {
struct VisibleBlock {
  void* ptr;
  size_t bytes;
  int device;
  bool in_use;
};
std::mutex g_visible_mu;
std::vector<VisibleBlock> g_visible;
}  // namespace

int tcpxuVisibleAlloc(int device, size_t bytes, void** host_ptr, void** dev_ptr) {
  if (!host_ptr || !dev_ptr || bytes == 0 || bytes > (64u << 20)) return TCPXU_INVALID_ARGUMENT;
  const char* sw = getenv("TCPXU_VISIBLE_DEVICE_MEMORY");
  if (sw && *sw == '0') {
    set_error("host-visible device memory is switched off (TCPXU_VISIBLE_DEVICE_MEMORY=0)");
    return TCPXU_INVALID_USAGE;
  }
  TCPXU_TRY(use_device(device));
  int large_bar = 0;
  if (hipDeviceGetAttribute(&large_bar, hipDeviceAttributeIsLargeBar, device) != hipSuccess || !large_bar) {
    set_error("device %d does not expose its memory to the host (no large BAR)", device);
    return TCPXU_INVALID_USAGE;
  }
  bytes = (bytes + 4095) / 4096 * 4096;
  std::lock_guard<std::mutex> lock(g_visible_mu);
  void* p = nullptr;
  for (auto& b : g_visible) {
    if (!b.in_use && b.device == device && b.bytes == bytes) {
      b.in_use = true;
      p = b.ptr;
      break;
    }
  }
  if (!p) {
    TCPXU_HIP(hipExtMallocWithFlags(&p, bytes, hipDeviceMallocFinegrained));
    g_visible.push_back(VisibleBlock{p, bytes, device, true});
  }
  memset(p, 0, bytes);  // the first host access: through the BAR, write-combined
  __builtin_ia32_sfence();
  *host_ptr = p;
  *dev_ptr = p;
  return TCPXU_SUCCESS;
}

int tcpxuVisibleFree(int device, void* host_ptr) {
  std::lock_guard<std::mutex> lock(g_visible_mu);
  for (auto& b : g_visible) {
    if (b.ptr == host_ptr && b.device == device && b.in_use) {
      b.in_use = false;
      return TCPXU_SUCCESS;
    }
  }
  set_error("not a block of tcpxuVisibleAlloc on device %d", device);
  return TCPXU_INVALID_ARGUMENT;
}

void tcpxuVisibleFlush(void) { __builtin_ia32_sfence(); }

static int launch_batch(const void* bounce_base, void* dst_base, const tcpxuLoadMeta* descs,
                        uint64_t n_descs, hipStream_t stream) {
  if (n_descs == 0) return TCPXU_SUCCESS;
  if (!bounce_base || !dst_base || !descs) {
    set_error("null pointer passed to unpack");
    return TCPXU_INVALID_ARGUMENT;
  }
  if (reinterpret_cast<uintptr_t>(descs) % 16 != 0) {
    set_error("descriptor array must be 16-byte aligned");
    return TCPXU_INVALID_ARGUMENT;
  }
  const bool short_list = n_descs <= kShortList;
  const uint32_t waves = short_list ? 1 : kLongListWaves;
  const void* kernel = short_list ? reinterpret_cast<const void*>(unpack_batch_kernel<1>) : reinterpret_cast<const void*>(unpack_batch_kernel<kLongListWaves>);
  uint64_t groups = (n_descs + waves - 1) / waves;
  // (A launch holds fewer than 2^32 threads: a list of more than 32 Mi descriptors takes several.)
  constexpr uint64_t kGroupsPerLaunch = 1ull << 23;
  for (uint64_t first = 0; first < groups; first += kGroupsPerLaunch) {
    uint32_t here = static_cast<uint32_t>(std::min(groups - first, kGroupsPerLaunch));
    void* args[] = {&bounce_base, &dst_base, &descs, &n_descs, &first, &here};
    TCPXU_HIP(hipLaunchKernel(kernel, dim3((here + 7) / 8 * 8), dim3(waves * kWaveLanes), args, 0, stream));
  }
  return TCPXU_SUCCESS;
}

int tcpxuUnpackBatch(int device, const void* bounce_base, void* dst_base, const tcpxuLoadMeta* descs,
                     uint64_t n_descs, void* stream) {
  TCPXU_TRY(use_device(device));
  return launch_batch(bounce_base, dst_base, descs, n_descs, static_cast<hipStream_t>(stream));
}

int tcpxuUnpackSlotNoAlloc(int device, const void* bounce_base, void* dst_base, const void* descs_dev,
                           uint32_t n_descs, void* done_flag_dev, uint64_t done_value, void* stream) {
  if (n_descs > TCPXU_SLOT_PAGES) {
    set_error("%u descriptors exceed the %d of one slot, the most this entry point serves", n_descs, TCPXU_SLOT_PAGES);
    return TCPXU_INVALID_ARGUMENT;
  }
  if (reinterpret_cast<uintptr_t>(done_flag_dev) % 8 != 0 || (done_flag_dev && done_value == 0)) {
    set_error("the completion word must be 8-byte aligned and its value nonzero");
    return TCPXU_INVALID_ARGUMENT;
  }
  if (n_descs > 0 && (!bounce_base || !dst_base || !descs_dev || reinterpret_cast<uintptr_t>(descs_dev) % 16 != 0)) {
    set_error("unpack needs bounce, destination and a 16-byte aligned descriptor address");
    return TCPXU_INVALID_ARGUMENT;
  }
  DeviceScope scope(device);
  TCPXU_TRY(scope.rc());
  hipStream_t s = static_cast<hipStream_t>(stream);
  // Without a completion word the end of the launch says everything.
  if (!done_flag_dev) return launch_batch(bounce_base, dst_base, static_cast<const tcpxuLoadMeta*>(descs_dev), n_descs, s);
  if (n_descs != 0 && n_descs <= kSmallSlot) {
    void* args[] = {&bounce_base, &dst_base, &descs_dev, &n_descs, &done_flag_dev, &done_value};
    TCPXU_HIP(hipLaunchKernel(reinterpret_cast<const void*>(unpack_small_slot_kernel), dim3(1), dim3(std::min(n_descs, kSmallSlotWaves) * kWaveLanes), args, 0, s));
    return TCPXU_SUCCESS;
  }
  TCPXU_TRY(launch_batch(bounce_base, dst_base, static_cast<const tcpxuLoadMeta*>(descs_dev), n_descs, s));
  void* args[] = {&done_flag_dev, &done_value};
  TCPXU_HIP(hipLaunchKernel(reinterpret_cast<const void*>(complete_slot_kernel), dim3(1), dim3(1), args, 0, s));
  return TCPXU_SUCCESS;
}

}  // extern "C"
