// Arrival counters of tiles that several workgroups finish together: which of them came last.
//
// A counter starts at zero; workgroup `part` of `parts` adds arrival_weight(part, parts), and the one whose sum is zero is
// the last. The weights of a launch add up to zero, so the counter is ready for the next launch without being cleared, and
// it is back at zero after any number of complete launches with any parts in any order of arrivals: launches that overlap on
// a counter by mistake spoil their own results only. (Counting up to `parts` and wrapping there, as atomicInc does, is exact
// for launches one after the other, but 2 and 4 parts interleaved can end at 4 and leave every later launch wrong.)
#pragma once

namespace rf {

// A proper subset of a launch's arrivals never adds up to zero: without part 0 its sum is its size, with part 0 it lacks the
// missing ones.
constexpr unsigned arrival_weight(unsigned part, unsigned parts) { return part == 0 ? 1u - parts : 1u; }

}  // namespace rf
