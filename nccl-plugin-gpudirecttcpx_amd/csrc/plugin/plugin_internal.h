// Internal types of the plugin library: the receive-side state that sits between the ncclNet_v7 calls and the
// GPU engine.  Everything here is host code; the GPU is reached only through the tcpxDeviceOps table.
//
// Roles (reference file:line in parentheses)
//   StageRing      fixed-capacity ring whose items move through an ordered list of stages
//                  (tcpxItemQueue, src/work_queue.h:78-130)
//   Request        one posted receive (tcpxRequest, src/work_queue.h:63-76) in a 16-deep RequestRing
//                  (tcpxRequestQueue, src/work_queue.h:174-212; states src/work_queue_states.h:30-39)
//   Task           one chunk of a request travelling on one data flow (tcpxTask, src/work_queue.h:38-59) in a
//                  6-deep TaskRing shared with the socket thread (tcpxTaskQueue, src/work_queue.h:132-172)
//   DataPipe       per-task staging of descriptors and page tokens (tcpxDataPipe, src/sock/datapipe.h:25-46)
//   DevmemSocket   synthetic stand-in for one devmem-TCP data socket
//   UnpackQueue    the slot ring in mapped memory (tcpxNetDeviceQueue, src/devcomm/unpack_defs1.h:39-74)
//   Comm           per-connection state (tcpxComm, src/common.h:159-216)
#ifndef TCPX_AMD_PLUGIN_INTERNAL_H_
#define TCPX_AMD_PLUGIN_INTERNAL_H_

#include <sched.h>
#include <sys/socket.h>
#include <sys/uio.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "tcpx_plugin.h"
#include "flow_mapper.h"
#include "trace.h"

namespace tcpx {

constexpr int kMaxRequests = 16;  // MAX_REQUESTS, src/work_queue.h:20
constexpr int kMaxTasks = 6;      // MAX_TASKS, src/work_queue.h:21
constexpr int kMaxFlows = 8;      // MAX_SOCKETS, src/macro.h:36
constexpr int kQueueDepth = NCCL_NET_DEVICE_UNPACK_MAX_QUEUE_DEPTH;
constexpr int kSlotPages = NET_UNPACK_MAX_SLICE_PAGES;
constexpr int kMaxDevices = 64;

constexpr int kOpSend = 0;  // TCPX_SOCKET_SEND
constexpr int kOpRecv = 1;  // TCPX_SOCKET_RECV

// Linux devmem-TCP control-message types the reference parses (src/sock/tcpx.h:30-42).
constexpr int kScmDevmemHeader = 98;
constexpr int kScmDevmemOffset = 99;

// ---- logging ------------------------------------------------------------------------------------------------------
void log_line(ncclDebugLogLevel level, unsigned long flags, const char* file, int line, const char* fmt, ...)
    __attribute__((format(printf, 5, 6)));
#define WARN(...) ::tcpx::log_line(NCCL_LOG_WARN, NCCL_ALL, __FILE__, __LINE__, __VA_ARGS__)
#define INFO(FLAGS, ...) ::tcpx::log_line(NCCL_LOG_INFO, (FLAGS), __FILE__, __LINE__, __VA_ARGS__)

// Propagate errors up (TCPXCHECK, src/misc/checks1.h:53-61).
#define TCPXCHECK(call)                                                    \
  do {                                                                     \
    ncclResult_t res_ = (call);                                            \
    if (res_ != ncclSuccess) {                                             \
      INFO(NCCL_ALL, "TCPXCHECK %s:%d -> %d", __FILE__, __LINE__, res_);   \
      return res_;                                                         \
    }                                                                      \
  } while (0)

// ---- StageRing ----------------------------------------------------------------------------------------------------
// Items enter at stage 0 and leave each stage in FIFO order.  `entered` counts items ever enqueued, `left[k]` items
// that have left stage k; an item leaving the last stage frees its slot.  Counters only grow, so
//   entered >= left[0] >= left[1] >= ... >= left[Stages-1]   and   entered - left[Stages-1] <= Capacity.
// With Counter = std::atomic<uint32_t> one thread may own `entered` and some stages while another owns the rest
// (single producer, single consumer per counter).
// A counter is written by exactly one thread: its new value is published with a release store and read with an
// acquire load (plain moves on x86; the default sequentially consistent store would be a locked exchange on every
// state transition of every task).
inline uint32_t counter_load(const uint32_t& c) { return c; }
inline void counter_store(uint32_t& c, uint32_t v) { c = v; }
inline uint32_t counter_load(const std::atomic<uint32_t>& c) { return c.load(std::memory_order_acquire); }
inline void counter_store(std::atomic<uint32_t>& c, uint32_t v) { c.store(v, std::memory_order_release); }

template <typename Item, int Capacity, int Stages, typename Counter>
struct StageRing {
  // Each counter has one writer and a cache line of its own: the stages of a task ring are advanced by two threads
  // (the socket thread and the proxy thread), and a counter that shared its line with the other thread's would be
  // taken away from its writer at every step of the other.
  struct alignas(64) Line {
    Counter v;
  };
  alignas(64) Counter entered;
  Line left_[Stages];  // left[k] of the description above
  alignas(64) Item items[Capacity];

  StageRing() {
    counter_store(entered, 0);
    for (int k = 0; k < Stages; ++k) counter_store(left_[k].v, 0);
  }
  uint32_t in_flight() const { return counter_load(entered) - counter_load(left_[Stages - 1].v); }
  bool empty() const { return in_flight() == 0; }
  uint32_t num_free() const { return Capacity - in_flight(); }
  bool has_free() const { return num_free() > 0; }
  Item* next_free() { return &items[counter_load(entered) % Capacity]; }
  void enqueue() { counter_store(entered, counter_load(entered) + 1); }

  uint32_t stage_begin(int k) const { return counter_load(left_[k].v); }
  uint32_t stage_end(int k) const { return k == 0 ? counter_load(entered) : counter_load(left_[k - 1].v); }
  bool has(int k) const { return stage_end(k) != stage_begin(k); }
  Item* first(int k) { return &items[stage_begin(k) % Capacity]; }
  void advance(int k) { counter_store(left_[k].v, counter_load(left_[k].v) + 1); }
};

// ---- unpack queue -------------------------------------------------------------------------------------------------
struct PageToken {  // struct devmemtoken / pgtok_t, src/devcomm/unpack_defs1.h:39-44
  uint32_t token_start;
  uint32_t token_count;
};

// Mapped host memory of one comm.  The prefix is NCCL's netUnpackMeta, bit for bit; the completion words that the
// GPU engine writes follow it.
struct QueueMeta {
  struct netUnpackMeta nccl;
  struct alignas(64) DoneWord {
    uint64_t value;
  } done[kQueueDepth];
};

struct QueueRecord {  // struct tcpxRecord, src/devcomm/unpack_defs1.h:46-51
  size_t flow_cnts[kQueueDepth];
  size_t pgtok_cnts[kQueueDepth][kMaxFlows];
  int flows[kQueueDepth][kMaxFlows];
  PageToken pgtoks[kQueueDepth][kMaxFlows][kSlotPages];
};

struct UnpackQueue {  // struct tcpxNetDeviceQueue, src/devcomm/unpack_defs1.h:53-59
  QueueMeta* meta = nullptr;      // host address
  QueueMeta* meta_dev = nullptr;  // device alias
  struct unpackNetDeviceHandle* dev_handle = nullptr;  // device memory
  union loadMeta* stage = nullptr;      // see QueueBlock
  union loadMeta* stage_dev = nullptr;
  uint64_t head = 0, tail = 0;
  int dev = 0;
  QueueRecord record;
};

struct UnpackSlot {  // struct unpackSlot, src/devcomm/unpack_defs1.h:61-74
  bool active = false;
  uint64_t idx = 0;
  union loadMeta* mem = nullptr;
  uint64_t* cnt = nullptr;  // nullptr also marks "no slot allocated yet" (src/net_tcpx.cc:890)
  uint64_t cnt_cache = 0;
  size_t* flow_cnt = nullptr;
  size_t* pgtok_cnts = nullptr;  // [kMaxFlows]
  int* flows = nullptr;          // [kMaxFlows]
  PageToken* pgtoks = nullptr;   // [kMaxFlows][kSlotPages]
};

ncclResult_t unpack_queue_new(int dev, bool passive, UnpackQueue** queue);
void unpack_queue_free(UnpackQueue* queue);
// src/devcomm/nccl/unpack1.h:30-65
void unpack_queue_next_free(UnpackQueue* queue, UnpackSlot* slot);

// ---- synthetic devmem socket --------------------------------------------------------------------------------------
struct DevmemVec {  // struct devmemvec, src/sock/tcpx.h:130-134
  uint32_t frag_offset;
  uint32_t frag_size;
  uint32_t frag_token;
};

// One control message as it lies in the buffer: the fields of struct cmsghdr, the vector, and the padding that the
// kernel zeroes too.
struct WireCmsg {
  size_t len;
  int level, type;
  DevmemVec v;
  uint32_t pad;
};
static_assert(sizeof(WireCmsg) == CMSG_SPACE(sizeof(DevmemVec)) && offsetof(WireCmsg, v) == CMSG_LEN(0) &&
                  offsetof(WireCmsg, level) == offsetof(struct cmsghdr, cmsg_level) &&
                  offsetof(WireCmsg, type) == offsetof(struct cmsghdr, cmsg_type),
              "one control message: header, 12 bytes, 4 of padding");
// The header (struct cmsghdr) of one that is not, or may not be, of that kind.  The same bytes are read both ways, so the
// compiler must not take the two for different memory.  (glibc's struct cmsghdr ends in a flexible array of characters, which
// says as much; other C libraries' do not.  Said of the header, which is read once a run: said of WireCmsg, which is written
// and read per fragment, it takes a bulk message 6 % longer, 307 -> 327 us for 256 MiB.)
struct __attribute__((may_alias)) CmsgHeader {
  size_t len;
  int level, type;
};
static_assert(sizeof(CmsgHeader) == sizeof(struct cmsghdr), "struct cmsghdr");

struct DataPipe {  // struct tcpxDataPipe, src/sock/datapipe.h:25-46
  std::vector<char> ctrl_data;           // control-message buffer handed to recvmsg
  std::vector<union loadMeta> scatter_list;  // [kSlotPages]
  union loadMeta* list;                      // where descriptors go: scatter_list
  uint64_t list_room = 0;                    // how many may go there: what fits, and fewer than kSlotPages of one chunk
  uint64_t cnt_cache = 0;
  uint64_t cnt_before = 0;  // descriptors of the same chunk that went into the slot before this pipe took over
  int bytes_cnt = 0;
  size_t* pgtok_cnt = nullptr;
  PageToken* pgtoks = nullptr;
  explicit DataPipe(bool own_list);  // false: without a scatter_list, for a pipe that is pointed at a slot
};

struct Comm;
struct DeviceState;

// The page references that the synthetic kernel keeps for one comm's sockets: each control message hands one to the
// receiver, SO_DEVMEM_DONTNEED gives it back (devmem TCP keeps a frag's reference with the socket that received it).
// The thread that receives writes `given`, the thread that consumes writes `back`, so a reference costs a load and a
// store and no locked instruction (with one counter per page and GPU that both threads and all comms updated, two
// locked ones per fragment were 9 of the 18.6 ns that a fragment of a bulk message cost the host).  Counted modulo 2^16:
// a comm holds at most kMaxRequests x kSlotPages = 2^15 references.
struct PageLedger {
  struct Page {
    uint16_t given, back;
  };
  // Written to by open(), so that a comm takes the page faults of its 4 bytes per page of arena when it is accepted and
  // not in its first receives (8 MiB of interleaved fragments from a 1 GiB arena, the first call of a fresh comm: 870 us of host
  // time without that, 160 with it, 90 once warm).
  Page* pages = nullptr;
  size_t n_pages = 0;
  // Both sides' totals, a line each for the thread that counts.
  alignas(64) std::atomic<uint64_t> given{0};
  alignas(64) std::atomic<uint64_t> back{0};

  bool open(size_t arena_pages);
  ~PageLedger() { free(pages); }
  uint64_t outstanding() const {
    const uint64_t returned = back.load(std::memory_order_acquire);  // (first: a page is given before it comes back)
    return given.load(std::memory_order_relaxed) - returned;
  }
  // Asks for a page's entry ahead of its use.  The token has not been checked yet, so the address is worked out as a number:
  // a pointer past the end of the block may not even be formed.
  void prefetch(uint32_t page) const {
    __builtin_prefetch(reinterpret_cast<const void*>(reinterpret_cast<uintptr_t>(pages) + sizeof(Page) * static_cast<size_t>(page)), 1);
  }
  // (Relaxed accesses to the two halves of an entry: a page comes back after the request that received it has gone
  // from one thread to the other through a task ring, which orders the two.)
  void give(uint32_t page) {
    uint16_t* g = &pages[page].given;
    __atomic_store_n(g, static_cast<uint16_t>(__atomic_load_n(g, __ATOMIC_RELAXED) + 1u), __ATOMIC_RELAXED);
  }
  bool take_back(uint32_t page) {  // false: not held, freed twice
    const uint16_t b = __atomic_load_n(&pages[page].back, __ATOMIC_RELAXED);
    if (b == __atomic_load_n(&pages[page].given, __ATOMIC_RELAXED)) return false;
    __atomic_store_n(&pages[page].back, static_cast<uint16_t>(b + 1u), __ATOMIC_RELAXED);
    return true;
  }
};

// One data flow's receive queue: what the kernel has for this socket.  recvmsg() hands out at most `max_bytes`
// and at most the control buffer's worth of fragments, one SCM_DEVMEM_OFFSET control message each, splitting a
// fragment when the byte budget ends inside it (the kernel does the same at the end of a recvmsg).
struct DevmemSocket {
  // Two sides.  Whoever delivers fragments appends to `arrived` under the lock; the one thread that receives on
  // this socket works on `rx`, which nobody else touches, and takes the lock only when `rx` has run empty, to swap
  // the two -- once per burst of deliveries instead of once per recvmsg.
  std::mutex mu;
  std::vector<tcpxSynthFrag> arrived;
  std::atomic<bool> any_arrived{false};  // `arrived` is not empty: a look at a quiet socket takes no lock
  std::vector<tcpxSynthFrag> rx;
  size_t head = 0;                     // read position in rx
  std::atomic<uint32_t> max_frags_per_recvmsg{0};  // 0 = no extra limit
  PageLedger* ledger = nullptr;        // the comm's page references
  void push(const tcpxSynthFrag* frags, size_t n);         // takes the lock
  void push_locked(const tcpxSynthFrag* frags, size_t n);  // the caller holds it
  ssize_t recvmsg(struct msghdr* msg, size_t max_bytes);
  // setsockopt(SO_DEVMEM_DONTNEED): gives page references back (src/sock/tcpx.h:299-307).
  int dontneed(const PageToken* tokens, size_t n);
};

// Walks the control messages of one recvmsg and appends one descriptor per devmem fragment to the pipe, coalescing
// consecutive page tokens (process_recv_cmsg, src/sock/tcpx.h:136-228).  Returns the bytes described, or -1 with
// *result set when the reference would have stopped the process.
ssize_t process_recv_cmsg(struct msghdr* msg, DataPipe* pipe, int offset, uint64_t dst_base_offset,
                          ncclResult_t* result);
// recvmsg + process_recv_cmsg for one task (gpudirectTCPXRecv, src/sock/tcpx.h:230-297).
ssize_t devmem_recv(DevmemSocket* sock, int size, int offset, DataPipe* pipe, uint64_t dst_base_offset,
                    ncclResult_t* result);

// ---- requests and tasks -------------------------------------------------------------------------------------------
struct Request;

// A task goes from the proxy thread (which fills it in) to the thread that serves its socket and back (descriptor
// count, result), and with a socket thread each direction is a cache line travelling between two CPUs: everything
// that travels is in the task's first line, and neither thread touches the other's bookkeeping (the pipe, the watch)
// on the way.
struct alignas(64) Task {  // struct tcpxTask, src/work_queue.h:38-59 (receive-side fields)
  int size = 0;
  int offset = 0;
  int request_offset = 0;
  uint8_t op = 0;
  bool started = false;  // its pipe has been set up
  uint16_t flow = 0;
  void* data = nullptr;
  Request* r = nullptr;
  ncclResult_t result = ncclSuccess;
  uint32_t cnt = 0;                // on the way out, descriptors of the chunk that are in the slot already; on the way
                                   // back, those the task produced (the pipe's cnt_cache when its last byte arrived)
  DataPipe* pipe = nullptr;        // the slot's own, for the life of the ring
  PageToken* pgtoks = nullptr;     // passive side: where the task's page tokens go (the request's slot, per flow)
  size_t* pgtok_cnt = nullptr;
  SlownessWatch watch;  // second line; recvmsg finding nothing, over and over (tcpxTask::timeout)
};
static_assert(offsetof(Task, watch) == 64, "what travels between the threads is one cache line");

enum TaskStage { kTaskActive = 0, kTaskCompleting = 1, kTaskInactive = 2, kTaskStages = 3 };
struct TaskRing : StageRing<Task, kMaxTasks, kTaskStages, std::atomic<uint32_t>> {
  // Where each slot's pipe keeps its descriptors, never written after construction: a line both threads can keep.
  alignas(64) const union loadMeta* scatter[kMaxTasks];
  TaskRing();
  ~TaskRing();
};

struct Request {  // struct tcpxRequest, src/work_queue.h:63-76
  Comm* comm = nullptr;
  void* data = nullptr;
  int op = 0;
  int mem_type = 0;
  int next_flow = -1;  // next_sock_id: >= 0 once a control message is pending for this request
  int next_size = 0;
  int offset = 0;
  int size = 0;          // the message's size once its first control message has been read; until then, posted_size
  int posted_size = 0;   // what irecv was given: the most the message may be
  int size_pending = 0;
  UnpackSlot slot;
  // Engine hand-off: the slot has been submitted, and the value its completion word will take.
  bool published = false;
  uint64_t done_value = 0;
  uint64_t published_ns = 0;
  SlownessWatch unpack_watch;  // the GPU holds the slot and the completion word does not come
};

enum RequestStage { kReqPosted = 0, kReqActive = 1, kReqTransmitting = 2, kReqInactive = 3, kReqStages = 4 };
using RequestRing = StageRing<Request, kMaxRequests, kReqStages, uint32_t>;

struct CtrlMessage {  // struct tcpxCtrl, src/common.h:127-133 (16 bytes on the wire)
  uint16_t type;
  uint16_t index;
  uint32_t size;
  uint32_t offset;
  uint32_t total;
} __attribute__((__packed__));
static_assert(sizeof(CtrlMessage) == 16, "control message is 16 bytes");

struct MemHandle {  // struct tcpxMemHandle, src/common.h:90-98
  void* ptr;
  size_t size;  // bytes registered (the reference does not keep it)
  int mem_type;
};

struct FlowData {  // struct tcpxFdData, src/common.h:144-157 (receive-side fields)
  DevmemSocket sock;
  TaskRing tasks;
  uint64_t bytes = 0;
  // struct tcpxSocketStats (receive side); the socket thread counts, the proxy thread reads.
  std::atomic<uint64_t> rx_ctrl_done_cnt{0}, rx_cnt{0}, rx_slow_cnt{0};
  // Each has one writer (the proxy thread, or the thread that runs this flow's socket), so a count is a load and a
  // store, not a locked read-modify-write.
  static void bump(std::atomic<uint64_t>& c) { c.store(c.load(std::memory_order_relaxed) + 1, std::memory_order_relaxed); }
};

struct Comm {  // struct tcpxComm, src/common.h:159-216
  bool passive = false;
  int dev = 0;
  int num_flows = 0;
  int end_flow_idx = 0;
  FlowData flows[kMaxFlows];
  PageLedger ledger;  // for the sockets of all flows
  std::unique_ptr<FlowScheduler> sched;  // tcpxComm::flow_mapper: the flows whose task ring has room
  std::mutex ctrl_mu;
  std::vector<CtrlMessage> ctrl_rx;  // the control socket's receive queue: what has arrived (under ctrl_mu)
  std::atomic<bool> ctrl_arrived{false};  // ctrl_rx is not empty: a look at a quiet control socket takes no lock
  std::vector<CtrlMessage> ctrl_local;  // ... and what the proxy thread has taken over from it, to read without the lock
  size_t ctrl_next = 0;                 // the first message of ctrl_local not yet read
  RequestRing rq;
  // The proxy thread's own view of what there is to do, so that a poll that finds nothing looks at nothing.
  uint32_t tasks_live = 0;    // tasks enqueued and not yet reaped, all flows
  uint32_t to_submit = 0;     // transmitting requests that the engine has not been given
  uint32_t submit_from = 0;   // ring position: every transmitting request before it has been given to the engine
  bool task_stats = false;       // task-level statistics are on
  bool receive_at_once = false;  // chunks whose bytes are there go straight into the slot (see receive_chunk)
  DataPipe direct{false};        // the pipe for that
  UnpackQueue* queue = nullptr;
  DeviceState* device = nullptr;
  uint64_t done_seq = 0;
  uint32_t slots_at_gpu = 0, max_slots_at_gpu = 0;  // slots submitted to the engine and not yet reported done
  SlownessWatch ctrl_watch;  // tcpxComm::ctrl_timeout
  uint64_t rx_ctrl_slow_cnt = 0, unpack_cnt = 0, unpack_slow_cnt = 0, unpack_ns = 0;
  std::unique_ptr<TraceBuffer> trace;  // tcpxComm::statsbuf; allocated when a stats level is on
  // Optional socket thread (persistentSocketThread, src/net_tcpx.cc:252-384).
  std::thread helper;
  std::atomic<bool> helper_stop{false};
  std::atomic<uint64_t> helper_cpus{0};  // CPUs the socket thread may run on, as it found them when it started
  bool use_helper = false;
};

// What tcpxListen writes into the caller's 128-byte handle and tcpxConnect_v5 reads back (the reference puts the
// listening socket's address there, src/connect.cc; with no sockets, the listener's identity does the same job).
struct ConnectHandle {
  uint64_t magic;  // kConnectMagic
  uint64_t id;     // the listener
  int32_t dev;
};
constexpr uint64_t kConnectMagic = 0x7463707861636365ull;  // "tcpxacce"
static_assert(sizeof(ConnectHandle) <= NCCL_NET_HANDLE_MAXSIZE, "the connect handle must fit NCCL's handle");

struct ListenComm {  // struct tcpxListenComm, src/common.h:112-124
  int dev;
  uint64_t id;
  // Connections made to this listener and not yet accepted (the listening socket's backlog).  connect() runs on
  // whichever thread the peer uses, accept() on the owner's.
  std::atomic<uint32_t> backlog;
};

// ---- per-GPU and global state -------------------------------------------------------------------------------------
struct QueueBlock {  // mapped metadata + device handle, recycled between comms (freed only when the engine is stopped)
  QueueMeta* meta;
  QueueMeta* meta_dev;
  struct unpackNetDeviceHandle* dev_handle;
  // Device memory the host can write, kStageDescs descriptors, or null: where the descriptors of a small request that has others
  // beside it, or of a longer one that is alone, are copied to as well, so that the GPU need not fetch them over PCIe (which
  // requests those are: descriptors_for_engine).
  union loadMeta* stage;
  union loadMeta* stage_dev;
};
constexpr uint32_t kStagedDescs = 16;   // a small request's, of which each slot has its own
constexpr uint32_t kAloneDescs = 512;   // of a longer request that is its comm's only one, behind the slots' own
constexpr uint32_t kStageDescs = kStagedDescs * kQueueDepth + kAloneDescs;

struct DeviceState {
  int dev = 0;
  std::mutex mu;
  void* arena = nullptr;
  size_t arena_bytes = 0;
  tcpxuEngine* engine = nullptr;
  bool engine_started = false;
  std::vector<Comm*> comms;           // open receive comms
  uint64_t pages_never_returned = 0;  // page references that comms still held when they were closed
  std::vector<QueueBlock> free_blocks;
  // What all comms have at the GPU, for a comm that asks whether its one small request has others beside it there: the sum of
  // their shares (see at_gpu_share).  On a line of its own: every comm's thread writes it.
  alignas(64) std::atomic<uint32_t> at_gpu{0};
};

// A comm's part of DeviceState::at_gpu by the slots that it has there.  All but the first count as kCrowd at once, so that a comm that
// keeps several there leaves the word alone.  kCrowd: the lists that a look of the engine brings along (the figures stand at
// descriptors_for_engine).
constexpr uint32_t kCrowd = 4;
constexpr uint32_t at_gpu_share(uint32_t slots) { return slots < 2 ? slots : kCrowd; }
inline void set_slots_at_gpu(Comm* comm, uint32_t slots) {
  const uint32_t was = at_gpu_share(comm->slots_at_gpu), is = at_gpu_share(slots);
  comm->slots_at_gpu = slots;
  if (is != was) comm->device->at_gpu.fetch_add(is - was, std::memory_order_relaxed);
}

// Who copies.  kDeviceHost: this plugin's engine unpacks every request and test() reports done after the copy; the
// plugin advertises an ordinary host-driven network (NCCL_NET_DEVICE_HOST), so no consumer kernel touches the
// queue.  kDeviceUnpack: the reference's division of labour -- the plugin only publishes descriptor counts
// (src/net_tcpx.cc:1354-1357), advertises NCCL_NET_DEVICE_UNPACK with the device handle, and the caller's kernel
// copies; the engine is never started.
constexpr int kDeviceHost = 0, kDeviceUnpack = 1;

struct Global {
  std::mutex mu;
  bool initialized = false;
  int device_type = kDeviceHost;  // NCCL_GPUDIRECTTCPX_AMD_DEVICE_TYPE=host|unpack
  std::mutex listen_mu;
  std::vector<ListenComm*> listeners;  // open listeners, for connect() to find by id
  ncclDebugLogger_t logger = nullptr;
  const tcpxDeviceOps* ops = nullptr;
  bool ops_injected = false;
  uint32_t carried_descs = 0;  // descriptors that the engine brings along with a submission (tcpxDeviceOps::engine_carried_descs)
  int n_devices = 0;
  DeviceState devices[kMaxDevices];
  // Flags (environment, range-checked in tcpxInit like TCPX_GET_INT_FLAG, src/net_tcpx.cc:440-452).
  int flows_per_comm = 4;
  int use_helper_thread = 0;
  int sched_alg = kSchedRoundRobin;  // NCCL_GPUDIRECTTCPX_SCHED_ALG
  bool fail_stop = true;
  // Observability (src/flags.cc:44-70, src/net_tcpx.cc:105-116).
  ClockFn clock = monotonic_ns;
  bool clock_injected = false;
  int64_t timeout_threshold_ns = 10000000000LL;  // 10 s
  int64_t timeout_frequency_ns = 30000000000LL;  // 30 s
  int slow_switch[kSlowKinds] = {0, 0, 0, 0};
  int slow_report[kSlowKinds] = {0, 0, 0, 0};
  int task_stats = 0;
  int request_stats = 0;
  int sampling_factor = 1;
  // NCCL_GPUDIRECTTCPX_RX_BINDINGS (struct tcpxBindings, src/common.h): CPUs for the socket threads of a device's comms.
  cpu_set_t rx_cpus[kMaxDevices];
  bool rx_bound[kMaxDevices] = {};
  char dev_names[kMaxDevices][32];
  char pci_paths[kMaxDevices][64];
};
extern Global g;

FlowScheduler* new_flow_scheduler(int alg);  // kSchedKaty, or round robin for anything else
int sched_alg_from_name(const char* name, bool* valid);  // "RR" / "KATY" (exact); anything else is round robin

// The synthetic peer and kernel, for drivers inside the library: many control messages under one lock, and the devmem
// contract (a fragment lies inside the arena and inside one 4 KiB page).
void ctrl_send_batch(Comm* comm, const CtrlMessage* messages, size_t n);
inline bool keeps_devmem_contract(const tcpxSynthFrag& f, size_t arena_bytes) {
  return static_cast<size_t>(f.frag_offset) + f.frag_size <= arena_bytes &&
         (f.frag_offset % SLICE_PAGE_SIZE) + f.frag_size <= SLICE_PAGE_SIZE;
}

const tcpxDeviceOps* default_device_ops();  // binds libtcpxu_hip.so, or nullptr (reason logged)
ncclResult_t device_result(int rc, const char* what);
// Called where the reference stops the process; honours tcpxSetFailStopForTesting.
ncclResult_t fail_stop(const char* what);

}  // namespace tcpx

#endif  // TCPX_AMD_PLUGIN_INTERNAL_H_
