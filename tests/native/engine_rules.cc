// The engine's decisions by numbers, at the numbers where they change (no GPU).
#include "engine_rules.h"

using namespace tcpxu;

// Of a grid with the leader and one worker on one compute unit, the rest are elsewhere: a worker that waits for enough of them
// must be able to see them come.
static_assert(!enough_can_be_elsewhere(2) && !enough_can_be_elsewhere(64), "small grids");
static_assert(!enough_can_be_elsewhere(257) && enough_can_be_elsewhere(258) && 258 - 2 == kEnoughElsewhere, "the line");
static_assert(enough_can_be_elsewhere(513), "two workers on each of 256 compute units");

int main() { return 0; }
