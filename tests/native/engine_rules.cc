// The engine's decisions by numbers, at the numbers where they change and against plain restatements (no GPU).
#include "engine_rules.h"

#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

using namespace tcpxu;

// Of a grid with the leader and one worker on one compute unit, the rest are elsewhere: a worker that waits for enough of them
// must be able to see them come.
static_assert(!enough_can_be_elsewhere(2) && !enough_can_be_elsewhere(64), "small grids");
static_assert(!enough_can_be_elsewhere(257) && enough_can_be_elsewhere(258) && 258 - 2 == kEnoughElsewhere, "the line");
static_assert(enough_can_be_elsewhere(513), "two workers on each of 256 compute units");

#define CHECK(c)                                                  \
  do {                                                            \
    if (!(c)) {                                                   \
      std::printf("line %d: %s does not hold\n", __LINE__, #c);   \
      return 1;                                                   \
    }                                                             \
  } while (0)

// A submission's ticket size, said with divisions; `burst` as the host marks it.
static uint32_t size_of(uint64_t in_flight, uint64_t n, uint64_t bytes, uint64_t workers, bool burst) {
  const double mean = bytes == 0 ? 4096.0 : static_cast<double>(bytes) / n;
  const uint32_t full = mean >= 2731 ? 16 : mean >= 2048 ? 32 : mean >= 1366 ? 48 : 64;
  if (burst) return full == 16 ? 18 : n > 1024 && n <= 1536 ? 48 : 32;
  if (n <= 16) return 16;
  if (in_flight >= 8 && n <= 32) return 32;
  const double per_worker = static_cast<double>(std::min<uint64_t>(in_flight * n, 1u << 20)) / workers;
  if (per_worker < 13) return 8;
  if (per_worker < 18) return 12;
  if (full == 16) return per_worker < 100 ? 14 : 16;
  return full == 48 && n <= 1024 && per_worker < 100 ? 32 : full;
}

// The leader before submissions of so many tickets each (none of more than the ring holds), workgroups finishing some of what is
// out between two of its passes: whether all of them are handed out, and never more tickets than the ring holds.  Entries are there
// as `there` says; when the next is not and everything is done, the leader sees that, as its looks do.  Now and then it takes those
// of one ticket in its rolling loop, which has a count of its own while tickets go on being finished.  The count that is read can
// lag behind what is done by a few tickets, also where the leader has seen that all is done: what it knows never goes back.
template <class There>
static bool all_handed_out(const std::vector<uint32_t>& tickets, uint32_t from, std::mt19937_64& rng, There there) {
  uint32_t out = from, done = from, known = from;
  size_t s = 0;
  auto counted = [&] { return done - static_cast<uint32_t>(rng() % 3 ? 0 : std::min<uint64_t>(rng() % 600, done - from)); };
  auto ask = [&] {
    const uint32_t before = known;
    known = known_done_after(known, counted());
    return known - before < 1u << 31 && done - known <= kTicketRing;
  };
  for (int waited = 0; waited < 100;) {
    const size_t before = s;
    bool here = false;
    while (rng() % 4 == 0) {
      const uint32_t own = counted();
      for (; s < tickets.size() && tickets[s] == 1 && there(s) && ticket_room(out, own) != 0; ++s) {
        ++out;
        if (rng() % 2 == 0 && done != out) ++done;
      }
      if (out - done > kTicketRing) return false;
    }
    if (ask_what_is_done(out, known, false) && !ask()) return false;
    while (s < tickets.size() && (here = there(s)) && tickets[s] <= ticket_room(out, known)) {
      out += tickets[s++];
      if (out - done > kTicketRing) return false;
    }
    if (s == tickets.size()) return true;
    if (s == before) {
      if (ask_what_is_done(out, known, here) && !ask()) return false;
      if (!here && done == out) known = out;
    }
    waited = s == before && done == out ? waited + 1 : 0;
    done += rng() % 4 == 0 ? out - done : static_cast<uint32_t>(rng() % (out - done + 1u));
  }
  return false;
}

int main() {
  for (const uint32_t done : {0u, 5u, 0u - 3u, 0u - kTicketRing}) {
    CHECK(ticket_room(done, done) == kTicketRing && ticket_room(done + 1, done) == kTicketRing - 1 && ticket_room(done + kTicketRing - 1, done) == 1);
    for (const uint32_t more : {0u, 1u, 5000u, kTicketRing, 1u << 30}) CHECK(ticket_room(done + kTicketRing + more, done) == 0);
  }
  for (const uint32_t known : {0u, 70000u, 0u - 2u}) {
    for (const uint32_t less : {0u, 1u, 600u, kTicketRing}) CHECK(known_done_after(known, known - less) == known);
    for (const uint32_t more : {1u, 600u, kTicketRing}) CHECK(known_done_after(known, known + more) == known + more);
  }
  std::mt19937_64 rng(1);
  const std::vector<std::vector<uint32_t>> lists = {{37500, 37500}, {1, kTicketRing}, {kTicketRing, kTicketRing, 1, kTicketRing}, {32768, 32769}, {32768, 32768, 32768}, {1, 65535, 2, 65534}};
  for (const auto& list : lists)
    for (const uint32_t from : {0u, 0u - 70000u, 0u - 3u}) CHECK(all_handed_out(list, from, rng, [](size_t) { return true; }));
  for (int i = 0; i < 3000; ++i) {
    std::vector<uint32_t> list(i % 100 == 0 ? 300000 : 1 + rng() % 200, 1u);
    for (uint32_t& t : list)
      if (list.size() < 300000 || rng() % 1000 == 0) t = 1 + static_cast<uint32_t>(rng() % (rng() % 3 ? 64 : kTicketRing));
    CHECK(all_handed_out(list, static_cast<uint32_t>(rng()), rng, [&](size_t) { return list.size() == 300000 || rng() % 8 != 0; }));
  }
  for (int i = 0; i < 2000000; ++i) {
    const uint32_t n = 1 + static_cast<uint32_t>(rng() % (rng() % 2 ? 3000 : 1u << 20)), in_flight = 1 + static_cast<uint32_t>(rng() % 300);
    const uint32_t workers = 1 + static_cast<uint32_t>(rng() % 1000);
    const uint64_t mean = rng() % 4200;  // (0: the caller did not say)
    const uint32_t bytes = static_cast<uint32_t>(std::min<uint64_t>(n * mean, 0xFFFFFFFFu));
    const bool marked = burst_of_pages(8, n, bytes, workers) || burst_of_short_fragments(8, n, bytes, workers);
    for (bool burst : {false, true})
      if (!burst || marked) CHECK(ticket_size_for_submission(in_flight, n, bytes, workers, burst) == size_of(in_flight, n, bytes, workers, burst));
    const uint32_t per = 1 + static_cast<uint32_t>(rng() % 64);
    CHECK(tickets_for(n, per) == (n + per - 1) / per);
  }
  // Bursts of short fragments (1800 bytes) on 512 workers: eight submissions or more, from 18 to fewer than 1000 descriptors per
  // worker in all, where fewer than 40 per worker are queued already.
  auto burst = [](uint32_t submissions, uint32_t n, uint32_t mean) { return burst_of_short_fragments(submissions, n, n * mean, 512); };
  CHECK(!burst(7, 1600, 1800) && burst(8, 1600, 1800));
  for (const uint32_t n : {1024u, 1025u, 1536u, 1537u})  // lengths between, of which the leader would write such tickets in another way
    CHECK(ticket_size_for_submission(16, n, n * 1800, 512, true) == (n == 1024 || n == 1537 ? 32u : 48u));
  CHECK(!burst(16, 575, 1800) && burst(16, 576, 1800));          // 18 x 512
  CHECK(burst(500, 1023, 1800) && !burst(500, 1024, 1800));      // 1000 x 512
  CHECK(burst(319, 1605, 1800) && !burst(320, 1600, 1800));
  CHECK(!burst(16, 1600, 1365) && burst(16, 1600, 1366) && burst(16, 1600, 2047) && !burst(16, 1600, 2048) && !burst(16, 1600, 0));
  CHECK(few_ahead_of_burst(0, 1u << 20, 1) && few_ahead_of_burst(12, 1706, 512) && !few_ahead_of_burst(12, 1707, 512));
  CHECK(!few_ahead_of_burst(UINT64_MAX / (1u << 20), 1u << 20, 512));
  std::puts("engine rules ok");
  return 0;
}
