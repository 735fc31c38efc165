// mci_fast_duo.hpp — launch interface of the single-coordinate chain with two waves a group of 64 walkers
// (mci_fast_duo.hip).
#pragma once

#include <cstdint>
#include <cstddef>

#include <hip/hip_runtime.h>

namespace mcid
{
struct FastArgs;

constexpr int DUO_CHUNK = 8; // steps of a ring half
inline size_t duo_lds(int d, bool x2)
{
    return 2 * DUO_CHUNK * 64 * 16 + sizeof(double) * (size_t)(x2 ? 2 : 1) * d * 64 + sizeof(double) * d + sizeof(float) * d;
}

// Whether a launch runs in this form (else on one wave a group, mci_fast.hip).  blocks: it sums blocks of
// B steps; shared_index: the index is the shared word's top bits.
// A producer wave is worth its barriers up to 16,384 walkers, one group a compute unit, and where the straight
// runs of eight and four steps are not cut too often.  Sampling, ms, one wave / two: shared index, 10,240 steps
// at d 16, 16,384 walkers, blocks of 160 1.42 / 1.27, blocks of 11 (704 steps) 0.16 / 0.19, 500 walkers at d 64,
// blocks of 17 0.33 / 0.41; an index drawn from a word of its own, whose second Philox block and product also
// go to the producer, 5,120 steps at d 10, 1,000 walkers, blocks of 20 1.81 / 1.49, blocks of 13 (832 steps) 0.198 /
// 0.191.  With more walkers two groups share a compute unit: as two workgroups their chain waves met on a
// SIMD (32,768 walkers 1.49 / 1.69), and two groups a workgroup wait for each other (blocks of 160 1.49 / 1.34,
// of 11 0.176 / 0.230).
inline bool duo_launch(int d, bool shared_index, bool blocks, int64_t B, int64_t W)
{
    return W <= 16384 && duo_lds(d, true) <= 160 * 1024 && (!shared_index || !blocks || B % 4 == 0 || B >= 256);
}

// one launch of kernel form fl (the F_* flags of mci_fast_dev.hpp: the native streams' block sums); false:
// there is no such form
bool launch_duo(int fl, const FastArgs &A, hipStream_t s);
} // namespace mcid
