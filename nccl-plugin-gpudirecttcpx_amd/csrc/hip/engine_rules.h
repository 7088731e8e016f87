// What the engine decides by numbers alone.  No device code and no HIP header: tests compile it on the host.
#ifndef TCPXU_ENGINE_RULES_H_
#define TCPXU_ENGINE_RULES_H_

#include <stdint.h>

namespace tcpxu {
namespace {

// The leader has its compute unit to itself.  Loads seem to return to a compute unit in the order in which it issued them,
// so the looks at the host's ring and the copy's loads wait for each other where both are under way.  A worker workgroup
// that finds itself there claims no ticket and leaves (its place then goes to the one workgroup of the grid that found
// none, which does the same) -- provided that this many others have started elsewhere: one that is placed while other
// kernels hold most of the GPU keeps all of its workers.  (Requests of 64 KiB: 2048 in one call 67.5 -> 63.5 us,
// 1024 41.4 -> 39.3, 16 to 256 within 2 % either way; a stream with 1024 in flight 40.5 -> 48.5 M/s, one comm's sixteen slots
// of 4 MiB 71.9 -> 72.5 % of the roofline; large requests the same, so two workers of 512 are not missed.)
constexpr uint32_t kEnoughElsewhere = 256;
// Whether a grid of so many workgroups can come to that many, with the leader and one worker on the leader's compute unit.  A
// smaller one neither asks where its workers are nor waits for others to start.
constexpr bool enough_can_be_elsewhere(uint32_t workgroups) { return workgroups >= kEnoughElsewhere + 2; }

}  // namespace
}  // namespace tcpxu
#endif  // TCPXU_ENGINE_RULES_H_
