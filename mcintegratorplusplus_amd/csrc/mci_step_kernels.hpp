// mci_step_kernels.hpp — the generic chain's kernels that evaluate sampling functions and
// observables: k_sample (MCI::sample: init + nsteps Metropolis steps + accumulation,
// MCIntegrator.cpp:252-321) and k_calibrate_indep (MCI::findMRT2Step, one independent loop per
// walker, MCIntegrator.cpp:87-168).  They are compiled into the library, and again, at run time,
// into a module with the caller's device functors (MCI_RTC_USER: the functor dispatch of
// mci_device.hpp is then defined ahead of this header).
#pragma once

#include "mci_kernels.hpp"

#include <float.h>

namespace mcid
{
// Where a walker's state lives.  LDSV: in the wave's LDS, one column a lane ([row][64]: xold, xnew, pold,
// pnew, and with observables their last values and running block sums), copied in at the start and out
// at the end of a launch; else in the chain's columns in HBM.  A step reads and writes most of the state
// several times with little arithmetic between, so the latency of those accesses bounds it: 16,384
// walkers of a three-component mixture in six dimensions took 17.9 us a step with block sums in HBM and
// take 6.3 us here (1,900 instructions, 160 of them branches, by the counters: one wave a SIMD, so their
// latency is not hidden).
constexpr int STATE_WAVE = 64;
constexpr size_t STATE_LDS_MAX = 80 * 1024;  // two waves a CU: beyond that the columns stay in HBM
// Waves a SIMD that a kind's registers leave room for.  In HBM a step waits for its accesses, so waves in
// flight count where there are more than one a SIMD (STATE_TWO walkers); the registers that the second one
// needs spill, which costs up to an eighth with fewer.  A call with 128 steps in 39 / 60 dimensions, one wave /
// two, ms: exp(-|x|), single-coordinate moves, 262,144 walkers 66.0 / 54.6, 65,536 29.2 / 32.8 (d 60).  In LDS it
// pays only for the long draws of the other distributions on the native streams (64 steps, d 4, 262,144 walkers:
// Student 78.1 / 61.2, gamma 66.1 / 51.6; the reference streams' Student 216 / 225, uniform moves 7.3 / 11.0).
constexpr int64_t STATE_TWO = 65536;
constexpr size_t STATE_LDS_TWO_MAX = 20 * 1024;  // eight waves a CU
inline __host__ __device__ constexpr int state_waves(int kind) { return kind == STATE_HBM_TWO || kind == STATE_LDS_TWO ? 2 : 1; }
inline __host__ __device__ constexpr bool state_in_lds(int kind) { return kind == STATE_LDS || kind == STATE_LDS_TWO; }
inline __host__ __device__ int state_rows(const Chain &c, int nobsdim) { return 2 * c.ndim + 2 * c.nproto + 2 * nobsdim; }
inline __host__ __device__ size_t state_lds(const Chain &c, int nobsdim)
{
    return sizeof(double) * STATE_WAVE * (size_t)state_rows(c, nobsdim) + sizeof(int) * STATE_WAVE * 2 * (size_t)c.nobs;
}
inline __host__ __device__ int chain_nobsdim(const Chain &c)
{
    int n = 0;
    for (int i = 0; i < c.nobs; ++i) { n += c.obs[i].nobs; }
    return n;
}

template <bool LDSV>
__device__ __forceinline__ Views state_views(const Chain &c, int64_t w, int nobsdim, double *lds)
{
    Views V;
    if constexpr (LDSV) {
        double *p = lds + threadIdx.x;
        auto next = [&](int rows) {
            const MciVec v{p, STATE_WAVE};
            p += rows * STATE_WAVE;
            return v;
        };
        V.xo = next(c.ndim);
        V.xn = next(c.ndim);
        V.po = next(c.nproto);
        V.pn = next(c.nproto);
        V.ov = next(nobsdim);
        V.sums = next(nobsdim);
        V.cnt = reinterpret_cast<int *>(lds + (int64_t)state_rows(c, nobsdim) * STATE_WAVE) + threadIdx.x;
        V.cs = STATE_WAVE;
        for (int i = 0; i < c.ndim; ++i) { V.xo[i] = c.xold[(int64_t)i * c.W + w]; }
    }
    else {
        V.xo = column(c.xold, c.W, w);
        V.xn = column(c.xnew, c.W, w);
        V.po = column(c.pold, c.W, w);
        V.pn = column(c.pnew, c.W, w);
        V.ov = column(c.obsval, c.W, w);
        V.sums = V.ov;
        V.cnt = nullptr;
        V.cs = 0;
    }
    return V;
}

template <bool LDSV>
__device__ __forceinline__ void state_back(const Chain &c, int64_t w, const Views &V)
{
    if constexpr (LDSV) {
        for (int i = 0; i < c.ndim; ++i) { c.xold[(int64_t)i * c.W + w] = V.xo[i]; }
    }
}

template <bool LDSV>
__device__ __forceinline__ void sample_walker(const Chain &c, int64_t nsteps, int accumulate_obs, int64_t w, double *lds)
{
    const int nobsdim = accumulate_obs ? chain_nobsdim(c) : 0;
    Lane L;
    load_lane(c, L, w);
    const Views V = state_views<LDSV>(c, w, nobsdim, lds);
    init_sampling(c, L, V);
    uint32_t dirty = 0xffffffffu;
    if (accumulate_obs) {
        if constexpr (LDSV) {
            for (int j = 0; j < nobsdim; ++j) { V.sums[j] = 0.0; }
            for (int i = 0; i < 2 * c.nobs; ++i) { V.cnt[i * V.cs] = 0; }
        }
        else { zero_accu(c, w); }
    }
    for (int64_t s = 0; s < nsteps; ++s) {
        if (c.npdf > 0) { step_mrt2<LDSV>(c, L, V); }
        else { step_random(c, L, V); }
        if (accumulate_obs) {
            accumulate<LDSV>(c, L, V, s, dirty);
            // file output (MCIntegrator.cpp:315-316, 509-516, 533-542): the last observable values
            // and the position after steps 0, f, 2f, ...
            if (c.rec_obs != nullptr && s % c.rec_fobs == 0) {
                const int64_t r = s / c.rec_fobs;
                for (int j = 0; j < c.rec_nobsdim; ++j) { c.rec_obs[(r * c.rec_nobsdim + j) * c.W + w] = V.ov[j]; }
            }
            if (c.rec_x != nullptr && s % c.rec_fx == 0) {
                const int64_t r = s / c.rec_fx;
                for (int i = 0; i < c.ndim; ++i) { c.rec_x[(r * c.ndim + i) * c.W + w] = V.xo[i]; }
            }
        }
    }
    if (accumulate_obs) {
        if constexpr (LDSV) {
            // Simple accumulators: one block, the whole run
            for (int i = 0; i < c.nobs; ++i) {
                const ObsDev &o = c.obs[i];
                if (o.acc != ACC_SIMPLE) { continue; }
                const double normf = 1. / (double)(1 + (nsteps - 1) / o.nskip);
                for (int j = 0; j < o.nobs; ++j) { o.data[(int64_t)j * c.W + w] = V.sums[o.voff + j] * normf; }
            }
        }
        else { finalize_accu(c, w, nsteps); }
    }
    state_back<LDSV>(c, w, V);
    store_lane(c, L);
}

template <int KIND>
__global__ __launch_bounds__(STATE_WAVE, state_waves(KIND)) void k_sample(Chain c, int64_t nsteps, int accumulate_obs,
                                                                          const uint8_t *active, const CalibCtrl *skip)
{
    extern __shared__ double state_sh[];
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= c.W) { return; }
    if (skip && skip->done) { return; }
    if (active && !active[w]) { return; }
    sample_walker<state_in_lds(KIND)>(c, nsteps, accumulate_obs, w, state_sh);
}

// step clamps of findMRT2Step (MCIntegrator.cpp:147-161)
__device__ inline void scale_and_clamp(const Chain &c, int64_t w, double fact, const double *dimSizes)
{
    const int64_t W = c.W;
    for (int t = 0; t < c.ntypes; ++t) { double &s = c.steps[(int64_t)t * W + w]; s = s * fact; }
    for (int i = 0; i < c.ndim; ++i) {
        int t = 0;
        while (t < c.ntypes && !(i < c.typeEnds[t])) { ++t; }
        double &s = c.steps[(int64_t)t * W + w];
        if (s > 0.5 * dimSizes[i]) { s = 0.5 * dimSizes[i]; }
    }
    for (int t = 0; t < c.ntypes; ++t) {
        double &s = c.steps[(int64_t)t * W + w];
        if (s < (double)FLT_MIN) { s = (double)FLT_MIN; }
    }
}

template <bool LDSV>
__device__ __forceinline__ void calibrate_walker(const Chain &c, int nfind, double target, int64_t min_stat, const double *dimSizes, int64_t w,
                                                 double *lds)
{
    Lane L;
    load_lane(c, L, w);
    const Views V = state_views<LDSV>(c, w, 0, lds);
    int cons = 0, counter = 0;
    while ((nfind < 0 && cons < 5) || counter < nfind) {
        init_sampling(c, L, V);
        for (int64_t s = 0; s < min_stat; ++s) { step_mrt2<LDSV>(c, L, V); }
        const double rate = (L.acc > 0) ? (double)L.acc / ((double)L.acc + (double)L.rej) : 0.;
        if (fabs(rate - target) < 0.05) { ++cons; }
        else { cons = 0; }
        const double fact = fmin(2., fmax(0.5, rate / target));
        scale_and_clamp(c, w, fact, dimSizes);
        L.st0 = c.steps[w];
        ++counter;
        if (nfind < 0 && counter >= -nfind) { break; }
    }
    state_back<LDSV>(c, w, V);
    store_lane(c, L);
}

template <int KIND>
__global__ __launch_bounds__(STATE_WAVE, state_waves(KIND)) void k_calibrate_indep(Chain c, int nfind, double target, int64_t min_stat,
                                                                                   const double *dimSizes)
{
    extern __shared__ double state_sh[];
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= c.W) { return; }
    calibrate_walker<state_in_lds(KIND)>(c, nfind, target, min_stat, dimSizes, w, state_sh);
}
} // namespace mcid
