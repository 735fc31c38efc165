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
// runs of eight and four steps are not cut too often.  Sampling (X2 and X2_SUM), ms, one wave / two: shared index,
// 16,384 walkers at d 16, 10,240 steps in blocks of 160 1.41 / 1.26, 704 in blocks of 11 0.169 / 0.179, 1,000
// walkers at d 2, 1,280 steps in blocks of 5 0.28 / 0.35; an index drawn from a word of its own, whose second
// Philox block and product also go to the producer, 1,000 walkers at d 10, 5,120 steps in blocks of 20 1.12 /
// 0.84, 832 in blocks of 13 0.206 / 0.187.  With more walkers two groups share a compute unit: as two workgroups
// their chain waves met on a SIMD (32,768 walkers 1.49 / 1.69), and two groups a workgroup wait for each other
// (blocks of 160 1.49 / 1.34, of 11 0.176 / 0.230).
inline bool duo_launch(int d, bool shared_index, bool blocks, int64_t B, int64_t W)
{
    return W <= 16384 && duo_lds(d, true) <= 160 * 1024 && (!shared_index || !blocks || B % 4 == 0 || B >= 256);
}

// one launch of kernel form fl (the F_* flags of mci_fast_dev.hpp: the native streams' block sums); false:
// there is no such form
bool launch_duo(int fl, const FastArgs &A, hipStream_t s);
} // namespace mcid
