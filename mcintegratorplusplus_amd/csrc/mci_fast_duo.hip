// mci_fast_duo.hip — single-coordinate moves on the native streams with two waves a group of 64 walkers.
//
// A chain wave alone on its SIMD spends about half of a step waiting (LDS reads, dependent FP64 operations,
// branches), and fills the waits with the next steps' Philox rounds (mci_fast.hip).  Where SIMDs are left
// over -- up to 16,384 walkers, a group a compute unit -- the words can come from a second wave instead: a producer wave draws
// eight steps ahead (coordinate, proposal, acceptance bits) into half of an LDS ring while the chain wave
// runs the eight steps in the other half; one barrier a half.
// Decisions, sums and their order are mci_fast.hip's, operation by operation.
//
// What bounds it: the chain wave's latency, about 120 ns a step without any Philox work (d 16, X2 and X2_SUM).
// Two things that lost: both screened decisions of a pair before one check for the exact test (1.63 against
// 1.56 ms for 65,536 walkers, four groups a workgroup), and a higher wave priority for the chain.
#include "mci_fast_dev.hpp"
#include "mci_fast_duo.hpp"

namespace mcid
{
namespace
{
constexpr int CH = DUO_CHUNK;

// what a step takes from its random words
struct __attribute__((aligned(16))) Draw
{
    double rr;      // proposal on (-1, 1)
    uint32_t slot;  // coordinate v's slot, 64 v + lane
    float u;        // the acceptance bits of the shared word
};

// the running sums of one walker (as Run64 of mci_fast.hip)
struct Run
{
    double r, Sr, Se, e, mult;
    uint32_t na;
};

// One step with draw D from its coordinate's value xo and block sum So, which the caller read and which
// hold the values after the step on return: mci_fast.hip's step64, operation by operation.
template <int FL>
__device__ __forceinline__ void step_duo(const FastArgs &A, double2 *rec, double *xs, const double *as, Run &R, const Draw &D, double &xo,
                                         double &So, float cv, uint64_t t, uint32_t wid, double step)
{
    constexpr bool HX2 = (FL & F_X2) != 0, HSUM = (FL & F_SUM) != 0, HEXP = (FL & F_EXP) != 0, ACC = (FL & 7) != 0, REC = HX2;
    const double xn = xo + step * D.rr;
    const double xn2 = xn * xn, xo2 = xo * xo;
    const double dx2n = xn2 - xo2;
    const float F = __builtin_amdgcn_exp2f(fmaf((float)dx2n, cv, A.uexp));
    const float Facc = fmaf(F, 0.9999f, -2.0f), Frej = F * 1.0001f;
    const bool acc = D.u < Facc;
    const bool band = !acc && D.u <= Frej;
    if (acc) { ++R.na; }
    double xsel = acc ? xn : xo, Snew = So;
    if (ACC) {
        const double dx2 = acc ? dx2n : 0.0;
        Snew = fma(dx2, R.mult, So);
        if (REC) { rec[D.slot] = make_double2(xsel, Snew); }
        else { xs[D.slot] = xsel; }
        R.r = R.r + dx2;
        if (!(HX2 && HSUM)) { R.Sr = fma(dx2, R.mult, R.Sr); }
        if (HEXP && acc) { const double en = exp(-(R.r / A.exp_div)); R.Se = R.Se + (en - R.e) * R.mult; R.e = en; }
    }
    else { xs[D.slot] = xsel; }
    if (__builtin_expect((__builtin_amdgcn_ballot_w64(D.u <= Frej) & ~__builtin_amdgcn_ballot_w64(acc)) != 0, 0)) {
        // the exact test: the shared word again, and the side-stream word below it
        uint32_t o0, o1, o2, o3, l0, l1, l2, l3;
        philox(0u, wid, (uint32_t)(t >> 1), (uint32_t)(t >> 33), A.key0, A.key1, o0, o1, o2, o3);
        philox(0x30000000u, wid, (uint32_t)t, (uint32_t)(t >> 32), A.key0, A.key1, l0, l1, l2, l3);
        const uint32_t w0 = pick((t & 1u) != 0, o2, o0);
        const uint64_t uw = (((uint64_t)w0 << 32) | l0) << A.ubits;
        const double u = (double)(uw >> 11) * 0x1p-53;
        const double av = as[D.slot / WAVE];
        const double ex = xn2 * av - xo2 * av;
        if (band && u <= exp(-ex)) {
            R.na += 1u;
            xsel = xn;
            if (ACC) {
                Snew = fma(dx2n, R.mult, So);
                if (REC) { rec[D.slot] = make_double2(xn, Snew); }
                else { xs[D.slot] = xn; }
                R.r = R.r + dx2n;
                if (!(HX2 && HSUM)) { R.Sr = fma(dx2n, R.mult, R.Sr); }
                if (HEXP) { const double en = exp(-(R.r / A.exp_div)); R.Se = R.Se + (en - R.e) * R.mult; R.e = en; }
            }
            else { xs[D.slot] = xn; }
        }
    }
    if (ACC) { R.mult = R.mult - 1.0; }
    xo = xsel;
    So = Snew;
}

template <int FL>
__global__ __launch_bounds__(2 * WAVE) void k_fast64_duo(FastArgs A)
{
    constexpr bool HX2 = (FL & F_X2) != 0, HSUM = (FL & F_SUM) != 0, HEXP = (FL & F_EXP) != 0, ACC = (FL & 7) != 0, REC = HX2;
    constexpr bool P2 = (FL & F_P2) != 0;
    extern __shared__ __attribute__((aligned(16))) double lds[];
    const int d = A.ndim, lane = threadIdx.x % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
    const bool producer = wave == 1;
    const int64_t w = (int64_t)blockIdx.x * WAVE + lane;
    const bool listed = w < A.W && (!A.wcount || w < *A.wcount);
    if (A.pend) {
        // the previous calibration iteration's factor, then nothing more once the loop has finished
        if (A.pend->apply && listed && !producer) {
            double st = A.steps[w] * A.pend->fact;
            for (int i = 0; i < d; ++i) {
                if (st > 0.5 * A.dimsizes[i]) { st = 0.5 * A.dimsizes[i]; }
            }
            if (st < (double)FLT_MIN) { st = (double)FLT_MIN; }
            A.steps[w] = st;
        }
        if (A.pend->done) { return; }
    }
    const bool live = listed && (!A.active || A.active[w]);
    if (__builtin_amdgcn_ballot_w64(live) == 0) { return; } // no walker here (the same 64 in both waves)
    // (lanes without a walker run along on a state of their own and store nothing: every wave reaches
    // every barrier)
    Draw *ring = reinterpret_cast<Draw *>(lds) + lane;  // [2][CH][64]
    double *state = lds + 2 * CH * WAVE * 2;
    double *as = state + (REC ? 2 : 1) * d * WAVE;
    float *cs = reinterpret_cast<float *>(as + d);
    for (int i = threadIdx.x; i < d; i += blockDim.x) {
        as[i] = A.a[i];
        cs[i] = (float)(-A.a[i] * 0x1.71547652b82fep+0);
    }
    const uint64_t t0 = live ? A.ctr[w] : 0;
    const uint32_t wid = live && A.wmap ? (uint32_t)A.wmap[w] : (uint32_t)w;
    const int64_t chunks = (A.nsteps + CH - 1) / CH;
    __syncthreads();
    if (producer) {
        // Pair tp of the native stream holds the words of steps 2 tp and 2 tp + 1.  A walker at an odd
        // step starts with the second half of its pair, and its pairs lie one step later in the ring.
        const bool odd = (t0 & 1u) != 0;
        const uint64_t base = (t0 >> 1) + (odd ? 1 : 0);
        auto draws = [&](uint64_t tp, Draw &a, Draw &b) {
            uint32_t o0, o1, o2, o3, p0 = 0u, p1 = 0u, g1, g3;
            philox(0u, wid, (uint32_t)tp, (uint32_t)(tp >> 32), A.key0, A.key1, o0, o1, o2, o3);
            if (!P2) { philox(1u, wid, (uint32_t)tp, (uint32_t)(tp >> 32), A.key0, A.key1, p0, g1, p1, g3); }
            auto make = [&](uint32_t shared, uint32_t next, uint32_t prop, uint64_t t) {
                uint32_t v, wp;
                if (P2) { v = __builtin_amdgcn_ubfe(shared, A.vshift, A.ibits); wp = next; }
                else { v = (uint32_t)draw_lemire(next, (uint32_t)A.nvecs, A.lemire_thr, wid, t, A.key0, A.key1); wp = prop; }
                Draw D;
                D.rr = fma((double)wp, 0x1p-31, -(1.0 - 0x1p-32));
                D.slot = v * WAVE + (uint32_t)lane;
                D.u = (float)(shared & A.umask);
                return D;
            };
            a = make(o0, o1, p0, 2 * tp);
            b = make(o2, o3, p1, 2 * tp + 1);
        };
        Draw carry, a, b;
        draws(t0 >> 1, a, carry);
        auto produce = [&](int64_t k) {
            Draw *half = ring + (k & 1) * (CH * WAVE) + (odd ? WAVE : 0);
            if (odd) { ring[(k & 1) * (CH * WAVE)] = carry; }
            const uint64_t tp = base + (uint64_t)k * (CH / 2);
#pragma unroll
            for (int j = 0; j < CH; j += 2) {
                draws(tp + j / 2, a, b);
                half[j * WAVE] = a;
                if (j + 2 < CH) { half[(j + 1) * WAVE] = b; }
                else if (odd) { carry = b; }
                else { half[(j + 1) * WAVE] = b; }
            }
        };
        produce(0);
        __syncthreads();
        for (int64_t k = 0; k < chunks; ++k) {
            if (k + 1 < chunks) { produce(k + 1); }
            __syncthreads();
        }
        return;
    }
    // the chain
    const int64_t B = A.blocksize;
    double2 *rec = reinterpret_cast<double2 *>(state); // X2: [d][64] {x_i, block sum of x_i^2}
    double *xs = state;                                // otherwise [d][64] x_i
    Run R{0.0, 0.0, 0.0, 0.0, (double)B, 0u};
    if (live) {
        for (int i = 0; i < d; ++i) {
            const double v = A.x64[(int64_t)i * A.W + w];
            if (REC) { rec[i * WAVE + lane] = make_double2(v, (double)B * (v * v)); }
            else { xs[i * WAVE + lane] = v; }
            R.r = R.r + v * v;
        }
    }
    else {
        for (int i = 0; i < (REC ? 2 : 1) * d; ++i) { state[i * WAVE + lane] = 0.0; }
    }
    const double step = live ? A.steps[w] : 0.0;
    if (ACC) { R.Sr = (double)B * R.r; }
    if (HEXP) { R.e = exp(-(R.r / A.exp_div)); R.Se = (double)B * R.e; }
    int64_t nacc = 0, b = 0, inblk = 0;
    // a block's end: its means out, |x|^2 recomputed exactly, the sums restarted (lanes without a walker
    // skip it whole: their numbers are not used)
    auto flush = [&]() {
        inblk = 0;
        ++b;
        if (!live) { return; }
        const double norm = 1. / (double)B;
        double rx = 0.0, sS = 0.0;
#pragma unroll 8
        for (int i = 0; i < d; ++i) {
            double v2;
            if (REC) {
                const double2 rv = rec[i * WAVE + lane];
                v2 = rv.x;
                sS = sS + rv.y;
                A.d_x2[((b - 1) * d + i) * A.W + w] = rv.y * norm;
                rec[i * WAVE + lane] = make_double2(v2, (double)B * (v2 * v2));
            }
            else { v2 = xs[i * WAVE + lane]; }
            rx = rx + v2 * v2;
        }
        if (HSUM) { A.d_x2sum[(b - 1) * A.W + w] = ((HX2 ? sS : R.Sr) * norm) / A.x2sum_div; }
        if (HEXP) { A.d_exp[(b - 1) * A.W + w] = R.Se * norm; }
        R.r = rx;
        R.Sr = (double)B * R.r;
        if (HEXP) { R.e = exp(-(R.r / A.exp_div)); R.Se = (double)B * R.e; }
        R.mult = (double)B;
    };
    auto single = [&](const Draw &D, int64_t s) {
        double x, S = 0.0;
        if (REC) { const double2 rv = rec[D.slot]; x = rv.x; S = rv.y; }
        else { x = xs[D.slot]; }
        step_duo<FL>(A, rec, xs, as, R, D, x, S, cs[D.slot / WAVE], t0 + (uint64_t)s, wid, step);
    };
    __syncthreads();
    for (int64_t k = 0; k < chunks; ++k) {
        const Draw *half = ring + (k & 1) * (CH * WAVE);
        const int64_t s0 = k * CH;
        const int n = (int)(A.nsteps - s0 < CH ? A.nsteps - s0 : CH);
        auto two = [&](const Draw &Da, const Draw &Db, int64_t s) {
            double xA, SA = 0.0, xB, SB = 0.0;
            if (REC) {
                const double2 ra = rec[Da.slot], rb = rec[Db.slot];
                xA = ra.x; SA = ra.y; xB = rb.x; SB = rb.y;
            }
            else { xA = xs[Da.slot]; xB = xs[Db.slot]; }
            const float cA = cs[Da.slot / WAVE], cB = cs[Db.slot / WAVE];
            step_duo<FL>(A, rec, xs, as, R, Da, xA, SA, cA, t0 + (uint64_t)s, wid, step);
            if (Db.slot == Da.slot) { xB = xA; SB = SA; } // the second step reads what the first wrote
            step_duo<FL>(A, rec, xs, as, R, Db, xB, SB, cB, t0 + (uint64_t)(s + 1), wid, step);
        };
        // straight on through the ring half where neither the run nor a block ends in it, else through four
        // or two steps where they can go together (branches cost a lone wave dearly: with a loop over the
        // pairs the 10,240 steps of 16,384 walkers took 1.73 ms instead of 1.27)
        if (n == CH && (!ACC || inblk + CH <= B)) {
            Draw D[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) { D[j] = half[j * WAVE]; }
#pragma unroll
            for (int j = 0; j < CH; j += 2) { two(D[j], D[j + 1], s0 + j); }
            inblk += CH;
            if (ACC && inblk == B) { flush(); }
        }
        else {
#pragma unroll 1
            for (int j = 0; j < n;) {
                const Draw *h = half + j * WAVE;
                const int64_t room = !ACC || B - inblk > n - j ? n - j : B - inblk; // >= 1
                if (room >= 4) {
                    two(h[0], h[WAVE], s0 + j);
                    two(h[2 * WAVE], h[3 * WAVE], s0 + j + 2);
                    j += 4;
                    inblk += 4;
                }
                else if (room >= 2) {
                    two(h[0], h[WAVE], s0 + j);
                    j += 2;
                    inblk += 2;
                }
                else {
                    single(h[0], s0 + j);
                    ++j;
                    ++inblk;
                }
                if (ACC && inblk == B) { flush(); }
            }
        }
        nacc += R.na;
        R.na = 0;
        __syncthreads();
    }
    if (!live) { return; }
    for (int i = 0; i < d; ++i) { A.x64[(int64_t)i * A.W + w] = REC ? rec[i * WAVE + lane].x : xs[i * WAVE + lane]; }
    A.ctr[w] = t0 + (uint64_t)A.nsteps;
    A.acc[w] = nacc;
    A.rej[w] = A.nsteps - nacc;
}

template <int FL>
bool launch(const FastArgs &A, hipStream_t s)
{
    const size_t sh = duo_lds(A.ndim, (FL & F_X2) != 0);
    hipLaunchKernelGGL(k_fast64_duo<FL>, dim3((unsigned)((A.W + WAVE - 1) / WAVE)), dim3(2 * WAVE), sh, s, A);
    return true;
}
} // namespace

bool launch_duo(int fl, const FastArgs &A, hipStream_t s)
{
    switch (fl) {
#define FORM(f) case f: return launch<f>(A, s);
        FORM(0) FORM(1) FORM(2) FORM(3) FORM(4) FORM(5) FORM(6) FORM(7)
        FORM(8) FORM(9) FORM(10) FORM(11) FORM(12) FORM(13) FORM(14) FORM(15)
#undef FORM
    default: return false;
    }
}
} // namespace mcid
