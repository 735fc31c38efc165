// mci_fast_group.hpp — launch interface of the kernels with a walker on a group of lanes
// (mci_fast_group.hip).
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace mcid
{
struct FastArgs;

// (lanes a walker, slots a lane) of the forms that are built.  Native streams: L S >= d + 1 words;
// reference streams: L S >= d coordinates.
#define GROUP_SHAPES(X)                                                                                  \
    X(2, 2) X(2, 4) X(2, 6) X(2, 10) X(2, 18) X(4, 2) X(4, 4) X(4, 6) X(4, 10) X(4, 14) X(4, 18) X(8, 10) X(8, 16)
#define GROUP_SHAPES_MT(X) X(4, 1) X(4, 2) X(4, 3) X(4, 4) X(4, 6) X(4, 8) X(4, 12) X(4, 16)

// The form for W walkers in d dimensions; false: none (the walker runs on one lane).
//  Reference streams: groups of four, up to 64 coordinates (elements 156 apart then share a lane).
//  Native streams: one wave per SIMD (1,024 in all) is the fewest that use the whole card, and a step
//  is shorter the more lanes share it, so the largest group that still gives at most one wave per
//  SIMD (d = 16, 16,384 walkers x 10,240 steps: one lane 7.9 ms, two 5.4, four 4.2), beyond that the
//  smallest that holds the walker in registers (d = 16, 65,536 walkers: one lane 8.0 ms, two 9.9, four
//  13.5; d = 35: two 5.0, four 5.3 for 2,560 steps): the ordered sum and the decision are then the
//  fewest.  Eight lanes measured the same as four for 1,000 walkers at d = 16, so they serve only the
//  widest walkers.
inline bool group_shape(bool mt, int d, int64_t W, int &L, int &S)
{
    if (W * (int64_t)d >= (int64_t)1 << 29) { return false; }  // a row of x_i^2 stays below 4 GiB
    constexpr int64_t FULL = 65536;                            // lanes of one wave per SIMD
    const int need = mt ? d : d + 1;
    const int lanes[] = {4, 2, 8};
    int bestL = 0, bestS = 0;
    auto smallest = [&](int l) {
        int s = 0;
#define SHAPE(a, b)                                                                                      \
    if (a == l && a * b >= need && (s == 0 || b < s)) { s = b; }
        if (mt) { GROUP_SHAPES_MT(SHAPE) }
        else { GROUP_SHAPES(SHAPE) }
#undef SHAPE
        return s;
    };
    if (mt) {
        L = 4;
        S = smallest(4);
        return S != 0;
    }
    for (int l : lanes) {
        const int s = smallest(l);
        if (s == 0) { continue; }
        if (l < 8 && W * l <= FULL) {
            L = l;
            S = s;
            return true;
        }
        if (bestL == 0 || l < bestL) {
            bestL = l;
            bestS = s;
        }
    }
    L = bestL;
    S = bestS;
    return bestL != 0 && d > 16;  // up to 16 coordinates one lane holds the walker
}

// The slots a lane for single-coordinate moves over d = 2^m coordinates on the reference streams (groups of
// four lanes, up to 64 coordinates); false: the walker runs on one lane
inline bool group_slots_vec(int d, int64_t W, int &S)
{
    S = d > 4 ? d / 4 : 1;
    return d <= 64 && (d & (d - 1)) == 0 && W * (int64_t)d < (int64_t)1 << 29;
}

// Whether such a launch of nsteps steps runs on groups of lanes; obs: the observables it sums or stores (the
// F_X2, F_SUM and F_EXP bits).  One lane a walker moves 72 bytes of generator state a step at up to 5.4 TB/s, and
// with x_i^2 a record of LDS for every coordinate; a group reads and writes the whole state once and issues
// its selects, and the ordered sum of sums and exponentials, on four times as many waves.
// ms of one launch, one lane / group:
//  without observables, 100 and 1,000 steps
//   16,384 walkers d 16 0.062 / 0.051, 0.54 / 0.26; d 64 0.066 / 0.073, 0.54 / 0.44
//   32,768 walkers d 16 0.065 / 0.064, 0.57 / 0.35; d 32 0.067 / 0.074, 0.57 / 0.45; d 64 0.071 / 0.132, 0.58 / 0.85
//   65,536 walkers d 16 0.081 / 0.120, 0.70 / 0.68; d 32 0.083 / 0.137, 0.70 / 0.85; d 64 0.088 / 0.250, 0.70 / 1.65
//  with x_i^2, sampling and estimation of traces at 65,536 walkers, 64 and 256 steps, one lane takes 0.7 to 0.9 and
//   1.0 to 1.4 times a group's time at d 1 to 64
//  |x|^2 alone, blocks of 16, 65,536 walkers, 1,024 steps: d 1 0.72 / 0.65, d 32 1.01 / 1.75, d 64 1.37 / 2.58;
//   exp(-|x|^2 / d) alone one lane takes 0.78 to 0.47 times a group's time
inline bool group_vec(int d, int64_t W, int64_t nsteps, int obs)
{
    constexpr int X2 = 1, EXP = 4;
    if (W <= 16384) { return true; }
    if (obs & X2) { return nsteps >= 128; }
    if (W <= 32768) { return d <= 16 || (d <= 32 && nsteps >= 512); }
    return nsteps >= 512 && !(obs & EXP) && d <= (obs ? 8 : 16);
}

// one launch of kernel form fl (the F_* flags of mci_fast_dev.hpp, without F_P2; vec: single-coordinate
// moves); false: there is no such form
bool launch_group_0(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
bool launch_group_1(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
bool launch_group_2(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
bool launch_group_3(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
bool launch_group_4(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
bool launch_group_5(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
bool launch_group_6(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s);
inline bool launch_group(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s)
{
    return launch_group_0(fl, vec, L, S, A, s) || launch_group_1(fl, vec, L, S, A, s) || launch_group_2(fl, vec, L, S, A, s) ||
           launch_group_3(fl, vec, L, S, A, s) || launch_group_4(fl, vec, L, S, A, s) || launch_group_5(fl, vec, L, S, A, s) ||
           launch_group_6(fl, vec, L, S, A, s);
}
} // namespace mcid
