// Synthetic devmem-TCP data socket and the descriptor builder that consumes it.
//
// The socket side produces exactly what the reference's receive path reads from the kernel: a msghdr whose
// control buffer holds one (SOL_SOCKET, SCM_DEVMEM_OFFSET) control message per fragment, each carrying a
// `struct devmemvec {frag_offset, frag_size, frag_token}` (src/sock/tcpx.h:130-134,157-181).  The builder side
// follows process_recv_cmsg (src/sock/tcpx.h:136-228) and gpudirectTCPXRecv (src/sock/tcpx.h:230-297).
#include <algorithm>

#include "plugin_internal.h"

namespace tcpx {

DataPipe::DataPipe(bool own_list)
    // 2048 control messages of CMSG_SPACE(sizeof(struct iovec)) bytes (src/devcomm/unpack_defs1.h:32-36).
    : ctrl_data(static_cast<size_t>(kSlotPages) * CMSG_SPACE(sizeof(struct iovec))), scatter_list(own_list ? kSlotPages : 0),
      list(scatter_list.data()) {}

void DevmemSocket::push(const tcpxSynthFrag* frags, size_t n) {
  std::lock_guard<std::mutex> lock(mu);
  push_locked(frags, n);
}

void DevmemSocket::push_locked(const tcpxSynthFrag* frags, size_t n) {
  if (n < 4) {  // (a range insert costs more than a few appends)
    for (size_t i = 0; i < n; ++i) arrived.push_back(frags[i]);
  } else {
    arrived.insert(arrived.end(), frags, frags + n);
  }
  any_arrived.store(!arrived.empty(), std::memory_order_release);
}

bool PageLedger::open(size_t arena_pages) {
  pages = static_cast<Page*>(calloc(arena_pages, sizeof(Page)));
  n_pages = pages ? arena_pages : 0;
  // One store to each page of it, through volatile so that it is not taken for what calloc has done already.
  constexpr size_t kEntriesPerHostPage = 4096 / sizeof(Page);
  for (size_t i = 0; i < n_pages; i += kEntriesPerHostPage) *static_cast<volatile uint16_t*>(&pages[i].given) = 0;
  if (n_pages != 0) *static_cast<volatile uint16_t*>(&pages[n_pages - 1].given) = 0;  // (the block need not start on a page)
  return pages != nullptr;
}

namespace {

constexpr size_t kPrefetchFrags = 8;  // page entries asked for ahead: the pages of a message lie anywhere in the arena

}  // namespace

ssize_t DevmemSocket::recvmsg(struct msghdr* msg, size_t max_bytes) {
  msg->msg_flags = 0;
  if (head == rx.size()) {  // everything taken over earlier has been received: look for new arrivals
    rx.clear();
    head = 0;
    if (any_arrived.load(std::memory_order_acquire)) {
      std::lock_guard<std::mutex> lock(mu);
      rx.swap(arrived);
      any_arrived.store(false, std::memory_order_relaxed);
    }
  }
  // A recvmsg that returns no bytes means "peer closed" to the caller, so empty fragments (which the adversarial
  // workload contains) only ever travel together with a non-empty one.
  auto payload_ahead = [&] {
    for (size_t i = head; i < rx.size(); ++i)
      if (rx[i].frag_size != 0) return true;
    return false;
  };
  bool payload = payload_ahead();  // (looks at one fragment unless empty ones are next)
  if (!payload && head < rx.size()) {
    // Only empty fragments are left on this side: the payload they travel with may have arrived meanwhile.
    {
      std::lock_guard<std::mutex> lock(mu);
      rx.insert(rx.end(), arrived.begin(), arrived.end());
      arrived.clear();
      any_arrived.store(false, std::memory_order_relaxed);
    }
    payload = payload_ahead();
  }
  if (!payload || max_bytes == 0) {
    msg->msg_controllen = 0;
    errno = EAGAIN;
    return -1;
  }
  const uint32_t limit = max_frags_per_recvmsg.load(std::memory_order_relaxed);
  uint32_t payload_left = limit != 0 ? limit : UINT32_MAX;
  WireCmsg* const first = static_cast<WireCmsg*>(msg->msg_control);
  WireCmsg* out = first;
  WireCmsg* const out_end = first + msg->msg_controllen / sizeof(WireCmsg);
  size_t bytes = 0;
  uint64_t refs = 0;
  tcpxSynthFrag* f = rx.data() + head;
  tcpxSynthFrag* const end = rx.data() + rx.size();
  const size_t n_pages = ledger->n_pages;
  if (limit == 0) {
    // Fragments that fit whole, without what only the last one needs to be asked.  (This loop, the one over messages in
    // process_recv_cmsg and the first case of dontneed: a fragment of a bulk message 6.4 -> 4.6 ns of host time.)
    for (const tcpxSynthFrag* const stop = f + std::min(end - f, out_end - out); f != stop && f->frag_size <= max_bytes - bytes; ++f) {
      *out++ = WireCmsg{CMSG_LEN(sizeof(DevmemVec)), SOL_SOCKET, kScmDevmemOffset, {f->frag_offset, f->frag_size, f->frag_token}, 0};
      bytes += f->frag_size;
      if (f->frag_token < n_pages) {
        ledger->give(f->frag_token);
        ++refs;
      }
      if (end - f > static_cast<ptrdiff_t>(kPrefetchFrags)) ledger->prefetch(f[kPrefetchFrags].frag_token);
    }
  }
  for (; f != end; ++f) {
    if (f->frag_size != 0) {
      if (bytes >= max_bytes || payload_left == 0) break;
      --payload_left;
    }
    if (out == out_end) {
      msg->msg_flags |= MSG_CTRUNC;
      break;
    }
    const uint32_t take = static_cast<uint32_t>(std::min<size_t>(f->frag_size, max_bytes - bytes));
    *out++ = WireCmsg{CMSG_LEN(sizeof(DevmemVec)), SOL_SOCKET, kScmDevmemOffset, {f->frag_offset, take, f->frag_token}, 0};
    bytes += take;
    // Every control message hands one page reference to the receiver.
    if (f->frag_token < ledger->n_pages) {
      ledger->give(f->frag_token);
      ++refs;
    }
    if (end - f > static_cast<ptrdiff_t>(kPrefetchFrags)) ledger->prefetch(f[kPrefetchFrags].frag_token);
    if (take != f->frag_size) {  // byte budget ended inside the fragment: the rest stays queued
      f->frag_offset += take;
      f->frag_size -= take;
      break;
    }
  }
  head = static_cast<size_t>(f - rx.data());
  ledger->given.store(ledger->given.load(std::memory_order_relaxed) + refs, std::memory_order_relaxed);
  msg->msg_controllen = static_cast<size_t>(out - first) * sizeof(WireCmsg);
  return static_cast<ssize_t>(bytes);
}

int DevmemSocket::dontneed(const PageToken* tokens, size_t n) {
  uint64_t given_back = 0;
  int rc = 0;
  for (size_t i = 0; i < n && rc == 0; ++i) {
    if (i + kPrefetchFrags < n) ledger->prefetch(tokens[i + kPrefetchFrags].token_start);
    if (tokens[i].token_count == 1 && tokens[i].token_start < ledger->n_pages && ledger->take_back(tokens[i].token_start)) {
      ++given_back;
      continue;
    }
    for (uint32_t k = 0; k < tokens[i].token_count; ++k) {
      const uint32_t page = tokens[i].token_start + k;
      if (page >= ledger->n_pages || !ledger->take_back(page)) {
        rc = -1;  // no such page, or freed twice
        break;
      }
      ++given_back;
    }
  }
  ledger->back.store(ledger->back.load(std::memory_order_relaxed) + given_back, std::memory_order_relaxed);
  return rc;
}

// The control message after `cm`, or null: the bounds of CMSG_NXTHDR, without the call into the C library that the
// macro makes for every message.
static inline CmsgHeader* next_cmsg(const struct msghdr* msg, CmsgHeader* cm) {
  const size_t at = static_cast<size_t>(reinterpret_cast<char*>(cm) - static_cast<char*>(msg->msg_control));
  const size_t left = msg->msg_controllen - at;
  if (cm->len < sizeof(CmsgHeader) || CMSG_ALIGN(cm->len) > left ||
      left - CMSG_ALIGN(cm->len) < sizeof(CmsgHeader))
    return nullptr;
  CmsgHeader* next = reinterpret_cast<CmsgHeader*>(reinterpret_cast<char*>(cm) + CMSG_ALIGN(cm->len));
  if (CMSG_ALIGN(next->len) > left - CMSG_ALIGN(cm->len)) return nullptr;  // runs past the end of the buffer
  return next;
}

ssize_t process_recv_cmsg(struct msghdr* msg, DataPipe* p, int offset, uint64_t dst_base_offset,
                          ncclResult_t* result) {
  int num_cm = 0;
  size_t host_bytes = 0;
  ssize_t dst_offset = 0;
  // What changes per fragment stays in registers: through `p` the compiler reads it back after every store.
  union loadMeta* const list = p->list;
  uint64_t cnt = p->cnt_cache;
  const uint64_t cnt_end = p->list_room;
  PageToken* const toks = p->pgtoks;
  size_t n_toks = *p->pgtok_cnt;
  uint32_t next_token = 0;  // the page that would continue the last run
  if (n_toks > 0) next_token = toks[n_toks - 1].token_start + toks[n_toks - 1].token_count;
  const uint64_t dst_base = static_cast<uint64_t>(offset) + dst_base_offset;
  const char* const control_end = static_cast<const char*>(msg->msg_control) + msg->msg_controllen;
  for (CmsgHeader* cm = reinterpret_cast<CmsgHeader*>(CMSG_FIRSTHDR(msg)); cm; cm = next_cmsg(msg, cm)) {
    // A run of devmem fragments as the kernel writes them, as many as there is room for: one comparison of the header each.
    const WireCmsg* w = reinterpret_cast<const WireCmsg*>(cm);
    const size_t room = std::min<size_t>({static_cast<size_t>(control_end - reinterpret_cast<const char*>(cm)) / sizeof(WireCmsg),
                                          static_cast<size_t>(cnt_end - cnt), static_cast<size_t>(kSlotPages) - n_toks});
    const WireCmsg* const w_end = w + room;
    for (; w != w_end && w->len == CMSG_LEN(sizeof(DevmemVec)) && w->level == SOL_SOCKET && w->type == kScmDevmemOffset; ++w) {
      const DevmemVec v = w->v;
      if (n_toks > 0 && next_token == v.frag_token) toks[n_toks - 1].token_count++;
      else toks[n_toks++] = PageToken{v.frag_token, 1};
      next_token = v.frag_token + 1u;
      union loadMeta& d = list[cnt++];
      d.src_off = v.frag_offset;
      d.len = v.frag_size;
      d.dst_off = static_cast<uint64_t>(dst_offset) + dst_base;
      dst_offset += v.frag_size;
    }
    if (const ptrdiff_t taken = w - reinterpret_cast<const WireCmsg*>(cm); taken != 0) {
      num_cm += static_cast<int>(taken);
      cm = next_cmsg(msg, reinterpret_cast<CmsgHeader*>(const_cast<WireCmsg*>(w - 1)));
      if (!cm) break;
    }
    if (cm->level != SOL_SOCKET || (cm->type != kScmDevmemOffset && cm->type != kScmDevmemHeader)) {
      INFO(NCCL_NET, "cmsg: unknown %u.%u", cm->level, cm->type);
      continue;
    }
    ++num_cm;
    DevmemVec v;
    memcpy(&v, reinterpret_cast<const char*>(cm) + CMSG_LEN(0), sizeof v);
    if (cm->type == kScmDevmemHeader) {
      // Payload that landed in host memory instead of a bounce page.  The reference has no working copy for it
      // (its gpu_inline_memcpy is a no-op, src/devcomm/nccl/inline.cu:48-60) and stops; so does this build.
      if (v.frag_size > 0) {
        host_bytes += v.frag_size;
        dst_offset += v.frag_size;
      }
      continue;
    }
    // Page tokens, run-length coded (src/sock/tcpx.h:190-199).
    if (n_toks > 0 && next_token == v.frag_token) {
      toks[n_toks - 1].token_count++;
    } else if (n_toks < static_cast<size_t>(kSlotPages)) {
      toks[n_toks++] = PageToken{v.frag_token, 1};
    } else {
      // The token list is the slot's, one per flow, and a request may put several chunks on one flow: it is full
      // when it holds as many runs as a slot holds descriptors.  (The reference zeroes the count per task and so
      // never gets here; it also forgets the earlier chunks' pages.)
      WARN("flow holds %zu page-token runs for one request, the most a slot records; failstop", n_toks);
      *p->pgtok_cnt = n_toks;
      *result = fail_stop("too many page-token runs on one flow of a request");
      return -1;
    }
    next_token = v.frag_token + 1u;
    if (cnt == cnt_end) {
      *p->pgtok_cnt = n_toks;
      const uint64_t of_chunk = cnt + 1 + p->cnt_before;
      if (of_chunk >= static_cast<uint64_t>(kSlotPages)) {  // src/sock/tcpx.h:183-187
        WARN("received %lu/%d segs, failstop", static_cast<unsigned long>(of_chunk), kSlotPages);
        *result = fail_stop("too many fragments in one task");
      } else {  // src/net_tcpx.cc:1350-1353
        WARN("request too many pages, one more than its slot had room for, failstop");
        *result = fail_stop("request needs more descriptors than a slot holds");
      }
      return -1;
    }
    // src/sock/tcpx.h:178-181: where the fragment lies in the bounce buffer, how long it is, and where in the
    // request's buffer it belongs: bytes of this recvmsg so far + bytes of the task so far + the task's offset in
    // the request.
    union loadMeta& d = list[cnt];
    d.src_off = v.frag_offset;
    d.len = v.frag_size;
    d.dst_off = static_cast<uint64_t>(dst_offset) + dst_base;
    cnt++;
    dst_offset += v.frag_size;
  }
  p->cnt_cache = cnt;
  *p->pgtok_cnt = n_toks;
  if (num_cm == 0) {  // src/sock/tcpx.h:202-209
    WARN("fatal, no cmsg");
    *result = fail_stop("recvmsg returned data without control messages");
    return -1;
  }
  if (dst_offset == 0) {  // src/sock/tcpx.h:210-217
    WARN("fatal, no data");
    *result = fail_stop("control messages describe no data");
    return -1;
  }
  if (host_bytes > 0) {  // src/sock/tcpx.h:218-225
    WARN("fatal, data landed on host memory");
    *result = fail_stop("payload landed in host memory");
    return -1;
  }
  return dst_offset;
}

ssize_t devmem_recv(DevmemSocket* sock, int size, int offset, DataPipe* p, uint64_t dst_base_offset,
                    ncclResult_t* result) {
  struct msghdr msg;
  struct iovec iov;
  memset(&msg, 0, sizeof msg);
  msg.msg_control = p->ctrl_data.data();
  msg.msg_controllen = p->ctrl_data.size();
  msg.msg_iov = &iov;
  msg.msg_iovlen = 1;
  iov.iov_base = nullptr;  // payload never lands in host memory here
  iov.iov_len = static_cast<size_t>(size - p->bytes_cnt);
  const ssize_t ret = sock->recvmsg(&msg, iov.iov_len);
  if (ret < 0) return ret;  // EAGAIN: nothing has arrived yet
  if (msg.msg_flags & MSG_CTRUNC) {  // src/sock/tcpx.h:267-274
    WARN("fatal, cmsg truncated, current msg_controllen %zu", p->ctrl_data.size());
    *result = fail_stop("control messages truncated");
    return -1;
  }
  const ssize_t described = process_recv_cmsg(&msg, p, offset, dst_base_offset, result);
  if (described < 0) return -1;
  if (described != ret) {  // src/sock/tcpx.h:276-283
    WARN("fatal, cmsg total bytes %zd, expected %zd", described, ret);
    *result = fail_stop("control messages do not add up to the bytes received");
    return -1;
  }
  p->bytes_cnt += static_cast<int>(ret);
  if (p->bytes_cnt >= size) p->bytes_cnt = 0;
  return ret;
}

TaskRing::TaskRing() {
  for (int i = 0; i < kMaxTasks; ++i) {
    items[i].pipe = new DataPipe(true);
    scatter[i] = items[i].pipe->scatter_list.data();
  }
}
TaskRing::~TaskRing() {
  for (int i = 0; i < kMaxTasks; ++i) delete items[i].pipe;
}

}  // namespace tcpx
