// The walk over a recvmsg's control messages and the synthetic recvmsg that fills them, against plain restatements of
// both: random mixtures of messages and fragments, with room for all of them and with less (no GPU).
#include <cstdio>
#include <random>
#include <vector>

#include "plugin_internal.h"

using namespace tcpx;

static std::mt19937_64 rng(12345);
static uint32_t below(uint32_t n) { return static_cast<uint32_t>(rng() % n); }
#define CHECK(c)                                                              \
  do {                                                                        \
    if (!(c)) {                                                               \
      std::printf("line %d, case %d: %s does not hold\n", __LINE__, at, #c);  \
      return false;                                                           \
    }                                                                         \
  } while (0)

// What process_recv_cmsg answers, said with the C library's macros and a step per message.
struct Answer {
  ssize_t rc = 0;
  std::vector<loadMeta> descs;
  std::vector<PageToken> toks;
};
static Answer walk(msghdr* msg, uint64_t room, std::vector<PageToken> toks, uint64_t base) {
  Answer a;
  a.toks = std::move(toks);
  int messages = 0;
  uint64_t bytes = 0, host = 0;
  for (cmsghdr* cm = CMSG_FIRSTHDR(msg); cm; cm = CMSG_NXTHDR(msg, cm)) {
    if (cm->cmsg_level != SOL_SOCKET || (cm->cmsg_type != kScmDevmemOffset && cm->cmsg_type != kScmDevmemHeader)) continue;
    ++messages;
    DevmemVec v;
    memcpy(&v, CMSG_DATA(cm), sizeof v);
    if (cm->cmsg_type == kScmDevmemHeader) {
      host += v.frag_size;
      bytes += v.frag_size;
      continue;
    }
    if (!a.toks.empty() && a.toks.back().token_start + a.toks.back().token_count == v.frag_token) ++a.toks.back().token_count;
    else if (a.toks.size() < static_cast<size_t>(kSlotPages)) a.toks.push_back(PageToken{v.frag_token, 1});
    else return a.rc = -1, a;
    if (a.descs.size() == room) return a.rc = -1, a;
    loadMeta d;
    d.src_off = v.frag_offset, d.len = v.frag_size, d.dst_off = base + bytes;
    a.descs.push_back(d);
    bytes += v.frag_size;
  }
  a.rc = messages == 0 || bytes == 0 || host != 0 ? -1 : static_cast<ssize_t>(bytes);
  return a;
}

static bool walk_case(int at) {
  const uint32_t n = 1 + below(40);
  alignas(16) static char control[64 * 64];
  memset(control, 0xEE, sizeof control);
  size_t len = 0;
  const uint32_t odd = below(3) == 0 ? 4 : 0;  // one message in four is something else, in a third of the cases
  uint32_t token = below(1000);
  for (uint32_t i = 0; i < n; ++i) {
    DevmemVec v{below(1u << 20), below(5) == 0 ? 0 : below(4097), token = below(3) == 0 ? below(1000) : token + 1};
    cmsghdr h{};
    size_t data = sizeof v;
    h.cmsg_level = SOL_SOCKET, h.cmsg_type = kScmDevmemOffset;
    if (odd != 0 && below(odd) == 0) {
      const uint32_t kind = below(5);
      if (kind == 0) h.cmsg_level = 41;                                   // somebody else's
      else if (kind == 1) h.cmsg_type = 7, data = 4 * below(8);           // unknown, of any length
      else if (kind == 2) h.cmsg_type = kScmDevmemHeader, v.frag_size = below(4) == 0 ? 100 : 0;
      else if (kind == 3) data = sizeof v + 4 + 4 * below(4);             // longer than the vector
      else h.cmsg_type = 7, data = 0;
    }
    h.cmsg_len = CMSG_LEN(data);
    memcpy(control + len, &h, sizeof h);
    if (data >= sizeof v) memcpy(control + len + CMSG_LEN(0), &v, sizeof v);
    len += CMSG_SPACE(data);
  }
  if (below(4) == 0) len -= std::min<size_t>(len, below(40));  // cut off anywhere in the last message
  msghdr msg{};
  msg.msg_control = control, msg.msg_controllen = len;
  const uint64_t before = below(4), room = before + (below(3) == 0 ? below(n + 1) : n + below(5));
  static PageToken toks[kSlotPages];
  size_t n_toks = below(4) == 0 ? kSlotPages - below(4) : below(3);
  for (size_t i = 0; i < n_toks; ++i) toks[i] = PageToken{static_cast<uint32_t>(5000 + 2 * i), 1};
  const uint64_t base = below(1u << 22);
  const Answer want = walk(&msg, room - before, std::vector<PageToken>(toks, toks + n_toks), 77 + base);
  DataPipe pipe(true);
  pipe.list_room = room, pipe.cnt_cache = before, pipe.pgtoks = toks, pipe.pgtok_cnt = &n_toks;
  ncclResult_t result = ncclSuccess;
  const ssize_t rc = process_recv_cmsg(&msg, &pipe, 77, base, &result);
  CHECK(rc == want.rc && (rc < 0) == (result != ncclSuccess));
  CHECK(n_toks == want.toks.size());
  for (size_t i = 0; i < n_toks; ++i) CHECK(toks[i].token_start == want.toks[i].token_start && toks[i].token_count == want.toks[i].token_count);
  if (rc < 0) return true;
  CHECK(pipe.cnt_cache == before + want.descs.size());
  for (size_t i = 0; i < want.descs.size(); ++i) {
    const loadMeta &a = pipe.list[before + i], &b = want.descs[i];
    CHECK(a.src_off == b.src_off && a.len == b.len && a.dst_off == b.dst_off);
  }
  return true;
}

// The socket: every fragment comes out in order and whole over a number of calls, none of which exceeds its byte budget,
// its control buffer or the socket's limit, or stops short of all three.
static bool socket_case(int at) {
  PageLedger ledger;
  CHECK(ledger.open(256));
  DevmemSocket sock;
  sock.ledger = &ledger;
  sock.max_frags_per_recvmsg = below(3) == 0 ? 1 + below(3) : 0;
  const uint32_t limit = sock.max_frags_per_recvmsg;
  std::vector<tcpxSynthFrag> frags(1 + below(60));
  for (auto& f : frags) f = tcpxSynthFrag{below(1u << 20), below(4) == 0 ? 0 : 1 + below(4096), below(300), 0};
  frags.back().frag_size = 17;  // (empty ones travel with payload behind them)
  sock.push(frags.data(), frags.size());
  std::vector<DevmemVec> got;
  size_t next = 0, done = 0;  // the fragment that comes next, and how much of it has come
  uint64_t refs = 0;
  while (next < frags.size()) {
    alignas(16) char control[32 * 64];
    msghdr msg{};
    msg.msg_control = control, msg.msg_controllen = 32 * (1 + below(64));
    const size_t room = msg.msg_controllen / 32, budget = 1 + below(9000);
    const ssize_t bytes = sock.recvmsg(&msg, budget);
    size_t sum = 0, payload = 0, messages = 0;
    if (bytes == 0) CHECK((msg.msg_flags & MSG_CTRUNC) != 0);  // a buffer full of empty fragments
    CHECK(bytes >= 0);
    for (cmsghdr* cm = CMSG_FIRSTHDR(&msg); cm; cm = CMSG_NXTHDR(&msg, cm)) {
      DevmemVec v;
      memcpy(&v, CMSG_DATA(cm), sizeof v);
      CHECK(cm->cmsg_level == SOL_SOCKET && cm->cmsg_type == kScmDevmemOffset && cm->cmsg_len == CMSG_LEN(sizeof v) && next < frags.size());
      const tcpxSynthFrag& f = frags[next];
      CHECK(v.frag_token == f.frag_token && v.frag_offset == f.frag_offset + done && done + v.frag_size <= f.frag_size);
      sum += v.frag_size, payload += v.frag_size != 0, ++messages;
      refs += f.frag_token < 256;
      done += v.frag_size;
      if (done == f.frag_size) ++next, done = 0;
    }
    CHECK(sum == static_cast<size_t>(bytes) && sum <= budget && messages <= room && (limit == 0 || payload <= limit));
    CHECK(next == frags.size() || sum == budget || messages == room || (limit != 0 && payload == limit));
    CHECK(((msg.msg_flags & MSG_CTRUNC) != 0) <= (messages == room));
  }
  CHECK(ledger.given.load() == refs && ledger.outstanding() == refs);
  // Given back singly and in runs; what was never given, or given back before, is refused.
  std::vector<uint32_t> held(256);
  for (size_t i = 0; i < 256; ++i) held[i] = ledger.pages[i].given;
  for (uint32_t page = 0; page < 256; ++page)
    for (; held[page] != 0; --held[page]) {
      PageToken run{page, 1};
      while (page + run.token_count < 256 && held[page + run.token_count] != 0 && below(2) == 0) --held[page + run.token_count++];
      CHECK(sock.dontneed(&run, 1) == 0);
    }
  CHECK(ledger.outstanding() == 0);
  const PageToken none{below(400), 1 + below(2)}, empty{3, 0};
  CHECK(sock.dontneed(&none, 1) != 0 && sock.dontneed(&empty, 1) == 0);
  return true;
}

// The walk reads the caller's buffer as headers and as WireCmsg in turn, and recvmsg writes it as the latter: what goes in one
// way must come out the other, whatever the compiler has inlined.
__attribute__((noipa)) static size_t written_as_wire(CmsgHeader* h, WireCmsg* w) {
  h->len = 1;
  w->len = 2;
  return h->len;
}
__attribute__((noipa)) static size_t written_as_header(CmsgHeader* h, WireCmsg* w) {
  w->len = 1;
  h->len = 2;
  return w->len;
}
static bool both_views_are_one_memory() {
  const int at = 0;
  alignas(16) static char control[sizeof(WireCmsg)];
  CHECK(written_as_wire(reinterpret_cast<CmsgHeader*>(control), reinterpret_cast<WireCmsg*>(control)) == 2);
  CHECK(written_as_header(reinterpret_cast<CmsgHeader*>(control), reinterpret_cast<WireCmsg*>(control)) == 2);
  return true;
}

int main() {
  tcpxSetFailStopForTesting(0);
  if (!both_views_are_one_memory()) return 1;
  for (int at = 0; at < 20000; ++at)
    if (!walk_case(at)) return 1;
  for (int at = 0; at < 3000; ++at)
    if (!socket_case(at)) return 1;
  std::puts("control messages ok");
  return 0;
}
