// mci_fast_plan.hpp — how the specialised kernels split a run into chunks, and the order in which the
// lane-group kernels make and take a generator's outputs.  Plain C++ with
// no HIP dependency (constexpr, so device code calls it too), so that the host-side tests can
// check the rules on runs far longer than a GPU test could take.
#pragma once

#include <cstdint>

namespace mcid
{
// Longest chunk the inner step loop runs (its counters are 32-bit).
constexpr int64_t FAST_MAX_CHUNK = (int64_t)1 << 30;

// Steps of the next chunk of a run of nsteps steps after s steps, inblk of them in the current
// block of B steps (B = nsteps for a Simple accumulator).  With accumulation (acc) a chunk never
// crosses a block end, so every block is flushed exactly when inblk reaches B; the result is in
// [1, 2^30] while s < nsteps.
constexpr int fast_chunk_len(int64_t nsteps, int64_t s, int64_t B, int64_t inblk, bool acc)
{
    int64_t lim = nsteps - s;
    if (acc && B - inblk < lim) { lim = B - inblk; }
    return (int)(lim < FAST_MAX_CHUNK ? lim : FAST_MAX_CHUNK);
}
// Bits of a native step's shared word (main word 0) that the index of a single-vector move over
// nvecs vectors takes: m when nvecs = 2^m with m <= 11 -- the FP64 acceptance uniform keeps the 53
// bits below them, the FP32 one (m <= 8) 24 -- else -1, and the index is drawn by Lemire's method
// from a word of its own.  Only the chain's own move shares (not one inside a MultiStepMove), and
// only in the native stream.
constexpr int shared_index_bits(bool philox, bool vec_move, bool multistep, int64_t nvecs)
{
    if (!philox || !vec_move || multistep || nvecs < 1 || (nvecs & (nvecs - 1)) != 0) { return -1; }
    int m = 0;
    while (((int64_t)1 << m) < nvecs) { ++m; }
    return m <= 11 ? m : -1;
}
// The FP32 chain shares only up to 8 bits (its 24-bit acceptance uniform sits below them).
constexpr int shared_index_bits32(int ibits) { return ibits <= 8 ? ibits : -1; }

// Steps between recomputations of |x|^2 from the position in the FP32 kernel.
constexpr int FAST32_REFRESH = 1024;

// Steps of the FP32 kernel's next chunk after s steps of nsteps, j of them in the current block of
// B (at most 2^31 - 1): at most FAST32_REFRESH, never past the block end.
constexpr int fast32_chunk_len(int64_t nsteps, int64_t s, int B, int j, bool acc)
{
    int64_t lim = nsteps - s;
    if (acc && (int64_t)(B - j) < lim) { lim = B - j; }
    return (int)(lim < FAST32_REFRESH ? lim : FAST32_REFRESH);
}

// The reference streams on groups of lanes: a generator's elements are twisted in MT_SEG parts of MT_CH,
// over and over, and a step takes `per` consecutive outputs (at most LEFT + 1) of a buffer of LEFT + MT_CH
// rows.  A part's outputs go to rows LEFT .. LEFT + MT_CH - 1, after the up to per - 1 that are left over,
// which move to the rows before LEFT, so that a step's outputs are always consecutive.
constexpr int MT_SEG = 6;
constexpr int MT_CH = 312 / MT_SEG;

// where a run ends: the next element of the round, and the outputs that were made but not taken (below
// per + MT_CH)
struct MtEnd
{
    int next, over;
};

// Runs nsteps steps: move(from, to, n) moves n outputs from rows from .. to rows to .., part(q) makes
// part q, step(row) takes the outputs from `row` on.  One count of all steps, whatever it is: parts follow
// each other without a break, since a part that began anew would twist elements out of their order.
template <int LEFT, class Move, class Part, class Step>
__attribute__((always_inline)) constexpr MtEnd mt_parts(int64_t nsteps, int per, Move move, Part part, Step step)
{
    int row = LEFT, wait = 0, next = 0;  // row of the next output, outputs waiting
    while (nsteps > 0) {
        // a round makes fewer steps than it holds outputs: its own count has 32 bits
        constexpr int ROUND = MT_SEG * MT_CH + LEFT;
        const int lim = nsteps < ROUND ? (int)nsteps : ROUND;
        int left = lim;
#pragma unroll
        for (int q = 0; q < MT_SEG; ++q) {
            if (left > 0) {
                move(row, LEFT - wait, wait);
                row = LEFT - wait;
                part(q);
                wait += MT_CH;
                next = (q + 1) * MT_CH;
                while (wait >= per && left > 0) {
                    const int first = row;
                    row += per;
                    wait -= per;
                    --left;
                    step(first);
                }
            }
        }
        nsteps -= lim - left;
    }
    return {next, wait};
}
} // namespace mcid
