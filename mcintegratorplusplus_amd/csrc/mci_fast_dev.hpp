// mci_fast_dev.hpp — what the specialised Metropolis kernels share: the launch arguments, the native
// stream's block function, and the reference streams' conversions.
#pragma once

#include "mci_f32math.hpp"
#include "mci_fast.hpp"
#include "mci_fast_plan.hpp"
#include "mci_kernels.hpp"

#include <float.h>

namespace mcid
{
constexpr int WAVE = 64;

struct FastArgs
{
    int64_t W;
    int ndim;
    int lanes;             // walkers of a wave (k_fast32)
    int64_t nsteps;
    uint32_t key0, key1;
    uint64_t *ctr;         // [W]
    double *x64;           // [ndim][W] (FP64 state, also FP32 mode's persistent copy)
    const double *a;       // [ndim] p_i = a_i x_i^2
    double *steps;         // [W] (one type; rescaled in place by a launch with a pending factor)
    int64_t *acc, *rej;    // [W]
    int64_t blocksize;     // B (Simple: nsteps)
    int64_t nblocks;
    double *d_x2;          // X2 data [nblocks][ndim][W] or nullptr
    double *d_x2sum;       // X2_SUM data [nblocks][1][W] or nullptr
    double *d_exp;         // EXP_X2 data [nblocks][1][W] or nullptr
    double *s_x2, *s_x2sum, *s_exp;  // Full accumulators: the sums of the traces, [ndim][W], [W], [W], or nullptr
    double x2sum_div;      // X2_SUM divisor
    double exp_div;        // EXP_X2 divisor
    int nvecs;
    uint32_t lemire_thr;   // 2^32 mod nvecs
    int ibits;             // index bits m in the shared word (nvecs = 2^m), -1: Lemire index
    int vshift;            // 32 - m: the index is the shared word's bits [vshift, 32) (none when m = 0)
    uint32_t ubits;        // max(m, 0): the acceptance uniform's bits start below the index
    uint32_t umask;        // FP64: the shared word's n = 32 - ubits acceptance bits
    float uexp;            // FP64: n, the screening exponent's offset
    const CalibCtrl *pend; // shared calibration: pending step factor, loop finished (FP64 kernel only)
    const double *dimsizes;
    uint64_t *mt;          // reference streams: [312][W] mt19937_64 states (F_MT launches)
    int32_t *mtp;          // [W] next state index
    const uint8_t *active; // [W] or nullptr: walkers whose flag is 0 do nothing (the independent
                           // decorrelation rounds of walkers that have finished theirs)
    const int32_t *wmap;   // or nullptr: the walker each lane's columns belong to (its Philox stream),
    const int32_t *wcount; // and the number of lanes in use, when the walkers are compacted
};

__device__ __forceinline__ void philox(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1,
                                       uint32_t &o0, uint32_t &o1, uint32_t &o2, uint32_t &o3)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r > 0) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = xor3((uint32_t)(p1 >> 32), c1, k0);
        const uint32_t n2 = xor3((uint32_t)(p0 >> 32), c3, k1);
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    o0 = c0; o1 = c1; o2 = c2; o3 = c3;
}

// a or b by a lane's flag as arithmetic on the values: a select of two elements of a register array
// can otherwise become a select of their addresses, which puts the array in scratch memory
__device__ __forceinline__ uint32_t pick(bool on, uint32_t a, uint32_t b) { return b ^ ((a ^ b) & (0u - (uint32_t)on)); }

// Lemire index on [0, range) from word w0 (SRRDVecMove.hpp:78 through uniform_int_distribution), for
// a range whose index the shared word does not hold: low = (w0 * range) mod 2^32 < thr = 2^32 mod
// range rejects and draws from the extra-word stream of step t.  thr is computed on the host; a wave
// vote skips the rare path.
__device__ __forceinline__ int draw_lemire(uint32_t w0, uint32_t range, uint32_t thr, uint32_t wid, uint64_t t, uint32_t k0, uint32_t k1)
{
    uint64_t prod = (uint64_t)w0 * range;
    if (__builtin_expect(__any((uint32_t)prod < thr), 0)) {
        uint32_t low = (uint32_t)prod;
        uint32_t kx = 0;
        while (low < thr) {
            const uint32_t k = 0x80000000u + (kx++);
            uint32_t o[4];
            philox(k >> 2, wid, (uint32_t)t, (uint32_t)(t >> 32), k0, k1, o[0], o[1], o[2], o[3]);
            prod = (uint64_t)o[k & 3u] * range;
            low = (uint32_t)prod;
        }
    }
    return (int)(prod >> 32);
}

// observable set of one launch (template flags: no per-step branches on them)
// F_P2: the index is the shared word's top bits (a power-of-two range); F_FULL: Full accumulators (every
// step's values stored)
// F_MT: the reference streams (mt19937_64 per walker) instead of the native ones
enum { F_X2 = 1, F_SUM = 2, F_EXP = 4, F_P2 = 8, F_FULL = 16, F_MT = 32 };

// canonical53 of the reference streams (generate_canonical<double, 53> on mt19937_64): w / 2^64,
// clamped below 1 (as in mci_device.hpp)
__device__ __forceinline__ double mt_canonical(uint64_t w)
{
    double r = (double)w / 18446744073709551616.0;
    if (r >= 1.0) { r = 0x1.fffffffffffffp-1; }
    return r;
}
} // namespace mcid
