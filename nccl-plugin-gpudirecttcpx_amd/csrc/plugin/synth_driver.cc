// tcpxSynthRunRequests: plays NCCL's receive proxy, the peer and the NIC for a list of requests, natively.
//
// The same sequence the reference's callers produce for the receive path -- irecv (src/net_tcpx.cc:921-944), one
// control message per chunk from the peer (struct tcpxCtrl, src/common.h:127-133), the chunk's fragments from
// the kernel (src/sock/tcpx.h:136-228), test() polled until done (src/net_tcpx.cc:1311-1374), iflush
// (src/net_tcpx.cc:946-954), irecvConsumed (src/net_tcpx.cc:1477-1543) -- with up to `window` requests posted at a time, as NCCL keeps several steps in
// flight.  Used by tests and by the benchmark to drive the plugin without an interpreter in the loop.
#include <time.h>

#include <mutex>
#include <vector>

#include "plugin_internal.h"

namespace tcpx {
namespace {

// The peer and the NIC for one posted request: the fragments of each flow's socket in arrival order (a socket keeps
// order only within itself, so handing each flow its fragments in one go is what many small deliveries come to), and
// one control message per chunk, in chunk order.  A chunk is a run of consecutive fragments on the same flow; an empty
// fragment cannot travel alone (recvmsg reports it together with payload), so it joins the run of the payload fragment
// before it, or after it at the very start.  One pass, each socket's lock taken once.
ncclResult_t feed_request(Comm* comm, const tcpxSynthFrag* frags, uint32_t n, uint32_t total, std::vector<CtrlMessage>* ctrl) {
  const uint32_t n_flows = static_cast<uint32_t>(comm->num_flows);
  const size_t arena = comm->device->arena_bytes;
  auto flow_of = [n_flows](const tcpxSynthFrag& f) { return f.flow < n_flows ? f.flow : f.flow % n_flows; };
  uint32_t first_payload = 0;
  while (first_payload < n && frags[first_payload].frag_size == 0) ++first_payload;
  if (first_payload == n) return ncclSuccess;
  ctrl->clear();
  {
    std::unique_lock<std::mutex> locks[kMaxFlows];
    uint32_t offset = 0, first = 0, bytes = 0;
    uint32_t flow = flow_of(frags[first_payload]);
    auto close_chunk = [&](uint32_t end) {
      DevmemSocket& sock = comm->flows[flow].sock;
      if (!locks[flow].owns_lock()) locks[flow] = std::unique_lock<std::mutex>(sock.mu);
      sock.push_locked(frags + first, end - first);
      ctrl->push_back(CtrlMessage{TCPX_CTRL_NORMAL, static_cast<uint16_t>(flow), bytes, offset, total});
      offset += bytes;
    };
    for (uint32_t i = 0; i < n; ++i) {
      const tcpxSynthFrag& f = frags[i];
      if (!keeps_devmem_contract(f, arena)) {
        WARN("fragment %u (offset %u, size %u) breaks the devmem contract", i, f.frag_offset, f.frag_size);
        return ncclInvalidArgument;
      }
      const uint32_t on = f.frag_size != 0 ? flow_of(f) : flow;
      if (on != flow) {
        close_chunk(i);
        flow = on;
        first = i;
        bytes = 0;
      }
      bytes += f.frag_size;
    }
    close_chunk(n);
  }
  ctrl_send_batch(comm, ctrl->data(), ctrl->size());
  return ncclSuccess;
}

double now_s() {
  struct timespec ts;
  clock_gettime(CLOCK_MONOTONIC, &ts);
  return static_cast<double>(ts.tv_sec) + 1e-9 * static_cast<double>(ts.tv_nsec);
}

}  // namespace
}  // namespace tcpx

using namespace tcpx;

extern "C" ncclResult_t tcpxSynthRunRequests(void* recvComm, const tcpxSynthFrag* frags, const tcpxSynthRequest* requests,
                                             uint32_t n_requests, void* dst_base, uint64_t dst_bytes, uint32_t window,
                                             uint32_t timeout_ms, double* seconds, double* latency_s) {
  Comm* comm = static_cast<Comm*>(recvComm);
  if (!comm || !comm->passive || !frags || !requests || !dst_base || window == 0 || window > static_cast<uint32_t>(kMaxRequests))
    return ncclInvalidArgument;
  if (dst_bytes > static_cast<uint64_t>(INT32_MAX)) dst_bytes = static_cast<uint64_t>(INT32_MAX);
  void* mhandle = nullptr;
  TCPXCHECK(tcpxRegMr(comm, dst_base, static_cast<int>(dst_bytes), NCCL_PTR_CUDA, &mhandle));
  struct Posted {
    void* request;
    double fed;
  };
  Posted posted[kMaxRequests];  // request i of the call at i % kMaxRequests
  std::vector<CtrlMessage> ctrl;
  uint32_t next = 0, oldest = 0;
  ncclResult_t rc = ncclSuccess;
  const double t0 = now_s();
  QuietTimeout quiet;
  while (rc == ncclSuccess && oldest < n_requests) {
    while (rc == ncclSuccess && next < n_requests && next - oldest < window) {
      const tcpxSynthRequest& r = requests[next];
      void* data = static_cast<char*>(dst_base) + r.dst_off;
      int size = static_cast<int>(r.bytes), tag = 0;
      Posted& p = posted[next % kMaxRequests];
      if ((rc = tcpxIrecv_v5(comm, 1, &data, &size, &tag, &mhandle, &p.request)) != ncclSuccess) break;
      rc = r.bytes == 0 ? tcpxSynthCtrlSend(comm, TCPX_CTRL_INLINE, 0, 0, 0, 0)
                        : feed_request(comm, frags + r.first_desc, r.n_descs, r.bytes, &ctrl);
      if (latency_s) p.fed = now_s();
      ++next;
    }
    if (rc != ncclSuccess) break;
    int done = 0, size = 0;
    void* request = posted[oldest % kMaxRequests].request;
    if ((rc = tcpxTest(request, &done, &size)) != ncclSuccess) break;
    if (done) {
      if (latency_s) latency_s[oldest] = now_s() - posted[oldest % kMaxRequests].fed;
      // NCCL's proxy flushes a finished receive before it hands the buffer on (iflush takes the request in the
      // request slot and answers with its size, src/net_tcpx.cc:946-954), then reports the slot consumed.
      const tcpxSynthRequest& fr = requests[oldest];
      void* fdata = static_cast<char*>(dst_base) + fr.dst_off;
      int fsize = -1;
      void* freq = request;
      if ((rc = tcpxIflush_v5(comm, 1, &fdata, &fsize, &mhandle, &freq)) != ncclSuccess) break;
      if (fsize != static_cast<int>(fr.bytes)) {
        WARN("iflush answered size %d for a request of %u bytes", fsize, fr.bytes);
        rc = ncclInternalError;
        break;
      }
      if ((rc = tcpxIrecvConsumed(comm, 1, request)) != ncclSuccess) break;
      ++oldest;
      quiet.reset();
    } else if (quiet.expired(1e-3 * timeout_ms, now_s)) {
      WARN("request %u did not complete within %u ms", oldest, timeout_ms);
      rc = ncclInternalError;
    }
  }
  if (seconds) *seconds = now_s() - t0;
  const ncclResult_t rc2 = tcpxDeregMr(comm, mhandle);
  return rc != ncclSuccess ? rc : rc2;
}
