// Order in which the work-groups of a causal grid take the tiles (no device code: plain constexpr functions).
#pragma once

namespace fa {

// An MI355X: 8 XCDs of 32 compute units.  (The order decides nothing but the time: on a device with another number the
// results are the same.)
constexpr int kXcds = 8, kCusPerXcd = 32;

// Place of work-group `slot` of `n` in a list of tiles sorted longest first, for a kernel that fits `per_cu`
// work-groups on each of `cus` compute units.  One to a CU, or a larger grid: the list as it is, whoever is done first
// takes the next longest.  A grid of at most two to a CU of a kernel that fits them starts all at once, so its order does
// not balance it but decides which two tiles share a CU: the first `cus` are the longest, longest first, the others
// follow shortest first.  B=1 H=16 M=N=4096 D=128 forward 0.086 -> 0.083 ms, B=4 H=8 M=N=1024 D=64 dQ 0.025 -> 0.023.
constexpr int causal_place(int slot, int n, int cus, int per_cu) {
    return per_cu >= 2 && n <= 2 * cus && slot >= cus ? n + cus - 1 - slot : slot;
}

}  // namespace fa
