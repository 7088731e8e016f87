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

// Launch-per-batch unpack: one wavefront per descriptor, four to a workgroup, as many workgroups as it takes.
//
// What bounds a short list is the chain launch -> descriptor -> payload -> store, each link a trip to memory; what
// bounds a long one is the memory system, and for short fragments how many wavefronts keep loads in flight.  Hence no
// LDS, no barrier and nothing carried from one fragment to the next: the descriptors go from the load into scalar
// registers, every wavefront of the 32 that a compute unit holds has a fragment of its own, and the dispatcher hands
// out new ones as they finish.  (Against workgroups of twelve wavefronts that staged their batch's descriptors in LDS,
// where a list of up to 8192 kept four of the twelve busy: 16 fragments 2.9 -> 2.4 us a launch (what the host needs for
// one), 4 MiB of wire fragments 5.1 -> 4.3 us, 8 MiB 6.6 -> 5.0, 16 MiB 10.0 -> 7.0, 64 MiB 23.6 -> 22.4; 256 MiB of
// 1.8 KiB fragments 126-140 -> 99 us = 5.4 TB/s r+w, which wants all 32 wavefronts: with 16 resident it takes 136 us.
// Whole pages by the half GiB move 2 % faster with 16 resident, 190 against 194 us; the list does not say which they
// are.  Half a fragment per wavefront, or two wavefronts to a workgroup, measured no better for short lists.)
constexpr uint32_t kBatchWaves = 4;
constexpr uint32_t kBatchThreads = kBatchWaves * kWaveLanes;
__global__ __launch_bounds__(kBatchThreads) __attribute__((amdgpu_waves_per_eu(8))) void unpack_batch_kernel(
    const uint8_t* __restrict__ bounce, uint8_t* __restrict__ dst, const tcpxuLoadMeta* __restrict__ descs,
    uint64_t n_descs, uint64_t first_group, uint32_t n_groups) {
  const uint32_t lane = threadIdx.x & (kWaveLanes - 1);
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWaveLanes)));
  // Neighbouring groups go to the same XCD: they share a destination line and, in mapped memory, the line that their
  // descriptors come in.
  const uint64_t group = xcd_contiguous_index(blockIdx.x, n_groups);
  if (group >= n_groups) return;
  const uint64_t i = (first_group + group) * kBatchWaves + wave;
  if (i < n_descs) copy_descriptor(bounce, dst, descs, n_descs, i, lane);
}

// One slot with a completion word (tcpxuUnpackSlotNoAlloc): the same, and the workgroup that finishes last writes the
// word.  Counting is two more trips to memory at the end of the chain; they are kept short by counting per workgroup in
// LDS first and, where many workgroups would queue up at one counter, in eight counters before the last (270 workgroups
// of a 4 MiB slot: 7.9 us a call with one counter, 6.4 with eight and one; 16 fragments: 4.5 and 4.9).  The last one at
// a counter sets it back to zero, so that the next call finds it as this one did.
constexpr uint32_t kSlotSubCounters = 8;
constexpr uint32_t kSlotOneCounterGroups = 64;  // workgroups up to which one counter is the faster way (69: even)
struct SlotCounters {
  struct alignas(128) Line {
    uint32_t count;
  };
  Line sub[kSlotSubCounters];
  Line top;
};
__global__ __launch_bounds__(kBatchThreads) __attribute__((amdgpu_waves_per_eu(8))) void unpack_slot_kernel(
    const uint8_t* __restrict__ bounce, uint8_t* __restrict__ dst, const tcpxuLoadMeta* __restrict__ descs,
    uint32_t n_descs, uint32_t n_groups, uint64_t* done_flag, uint64_t done_value, SlotCounters* counters) {
  __shared__ uint32_t waves_done;
  const uint32_t lane = threadIdx.x & (kWaveLanes - 1);
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWaveLanes)));
  if (threadIdx.x == 0) waves_done = 0;
  __syncthreads();
  const uint32_t group = static_cast<uint32_t>(xcd_contiguous_index(blockIdx.x, n_groups));
  const uint32_t i = group * kBatchWaves + wave;
  if (group < n_groups && i < n_descs) copy_descriptor(bounce, dst, descs, n_descs, i, lane);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this wavefront's write-through stores are acknowledged
  if (lane != 0) return;
  // Every count is a read-modify-write at agent scope that follows the acknowledgement of the stores it stands for.
  auto last_at = [](uint32_t* counter, uint32_t of) {
    if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != of) return false;
    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  };
  if (__hip_atomic_fetch_add(&waves_done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + 1u != kBatchWaves) return;
  uint32_t at_top = gridDim.x;
  if (n_groups > kSlotOneCounterGroups) {
    // The grid is a multiple of eight workgroups, so each of the eight counters has an eighth of them.
    static_assert(kSlotSubCounters == 8, "the grid is rounded up to a multiple of eight");
    if (!last_at(&counters->sub[blockIdx.x % kSlotSubCounters].count, gridDim.x / kSlotSubCounters)) return;
    at_top = kSlotSubCounters;
  }
  if (last_at(&counters->top.count, at_top)) __hip_atomic_store(done_flag, done_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// An empty slot: nothing to copy, only the word.
__global__ void complete_empty_slot_kernel(uint64_t* done_flag, uint64_t done_value) {
  __hip_atomic_store(done_flag, done_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The counters, in a fixed array of device memory: a set for each of kSlotCalls calls in turn, so that calls may overlap
// on a GPU (two streams, a call beside a replayed graph) unless two whose kernels run at the same time were made a multiple
// of that many apart.  1024, so that a stream which falls behind, or a graph, meets that by no ordinary chance; 64 measured
// the same (a 4 MiB slot 6.15 us a call).  In host code the name is only a handle for hipGetSymbolAddress; kernels get the
// address it returns.
constexpr uint32_t kSlotCalls = 1024;
static __device__ SlotCounters slot_counters[kSlotCalls];

struct DeviceProps {
  bool valid = false;
  int compute_units = 0;
  char name[256] = "";
};
DeviceProps g_props[kMaxDevices];

}  // namespace

int use_device(int device) {
  if (device < 0 || device >= kMaxDevices) {
    set_error("device index %d out of range", device);
    return TCPXU_INVALID_ARGUMENT;
  }
  TCPXU_HIP(hipSetDevice(device));
  if (!g_props[device].valid) {
    hipDeviceProp_t p;
    TCPXU_HIP(hipGetDeviceProperties(&p, device));
    g_props[device].compute_units = p.multiProcessorCount;
    snprintf(g_props[device].name, sizeof g_props[device].name, "%s (%s)", p.name, p.gcnArchName);
    g_props[device].valid = true;
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
  uint64_t groups = (n_descs + kBatchWaves - 1) / kBatchWaves;
  // (A launch holds fewer than 2^32 threads: a list of more than 32 Mi descriptors takes several.)
  constexpr uint64_t kGroupsPerLaunch = 1ull << 23;
  for (uint64_t first = 0; first < groups; first += kGroupsPerLaunch) {
    uint32_t here = static_cast<uint32_t>(std::min(groups - first, kGroupsPerLaunch));
    void* args[] = {&bounce_base, &dst_base, &descs, &n_descs, &first, &here};
    TCPXU_HIP(hipLaunchKernel(reinterpret_cast<const void*>(unpack_batch_kernel), dim3((here + 7) / 8 * 8), dim3(kBatchThreads), args, 0, stream));
  }
  return TCPXU_SUCCESS;
}

int tcpxuUnpackBatch(int device, const void* bounce_base, void* dst_base, const tcpxuLoadMeta* descs,
                     uint64_t n_descs, void* stream) {
  TCPXU_TRY(use_device(device));
  return launch_batch(bounce_base, dst_base, descs, n_descs, static_cast<hipStream_t>(stream));
}

// The address of the counters on each device, asked for once per device with that device current.
static std::atomic<SlotCounters*> g_slot_counters[kMaxDevices];
static std::atomic<uint32_t> g_slot_calls[kMaxDevices];

static int next_slot_counters(int device, SlotCounters** out) {
  SlotCounters* all = g_slot_counters[device].load(std::memory_order_acquire);
  if (!all) {  // (two threads may both ask; they get the same answer)
    void* p = nullptr;
    TCPXU_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(slot_counters)));
    if (!p) {
      set_error("the slot counters have no address on device %d", device);
      return TCPXU_INTERNAL_ERROR;
    }
    all = static_cast<SlotCounters*>(p);
    g_slot_counters[device].store(all, std::memory_order_release);
  }
  *out = all + g_slot_calls[device].fetch_add(1, std::memory_order_relaxed) % kSlotCalls;
  return TCPXU_SUCCESS;
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
  if (n_descs == 0) {
    void* args[] = {&done_flag_dev, &done_value};
    TCPXU_HIP(hipLaunchKernel(reinterpret_cast<const void*>(complete_empty_slot_kernel), dim3(1), dim3(1), args, 0, s));
    return TCPXU_SUCCESS;
  }
  SlotCounters* counters = nullptr;
  TCPXU_TRY(next_slot_counters(device, &counters));
  uint32_t groups = (n_descs + kBatchWaves - 1) / kBatchWaves;
  void* args[] = {&bounce_base, &dst_base, &descs_dev, &n_descs, &groups, &done_flag_dev, &done_value, &counters};
  TCPXU_HIP(hipLaunchKernel(reinterpret_cast<const void*>(unpack_slot_kernel), dim3((groups + 7) / 8 * 8), dim3(kBatchThreads), args, 0, s));
  return TCPXU_SUCCESS;
}

}  // extern "C"
