// mci_fast_group.hip — Metropolis kernels with a walker's coordinates spread over a group of lanes (FP64,
// one diagonal Gaussian or exp(-|x|^2), unbounded domain, observables as in mci_fast.hip): all-coordinate
// moves on both random streams (SRRDAllMove with one step size, MoveType::All, the reference's default
// move), and single-coordinate moves on the reference streams (k_fast64_vec4, below).
//
// k_fast64_grp: a step proposes every coordinate, x'_i = x_i + step r_i, sums the protos (x'_i x'_i) a_i in coordinate
// order and tests u <= exp(sum p - sum p'), with the screen of k_fast64.  Every operation and its order
// are those of the generic kernel, so every number is bit-identical to it.
//
// What bounds it is instruction issue: a step's instructions divide over the group's lanes (Philox
// blocks or generator elements, proposals, squares, block sums), all but the ordered sum and the
// decision, which every lane repeats.  A whole walker on one lane needs its state in LDS beyond 16
// coordinates (one wave per CU at d = 50: 32.2 ms for 20,011 walkers x 2,560 steps) and, on the
// reference streams, reads and writes 24 bytes of generator state in HBM for every output (12.5 ms
// for 65,536 walkers x 2,048 traced steps at d = 16).  On groups of four the coordinates stay in
// registers (4.4 ms) and so do the 312 generator elements, 78 a lane, loaded once per launch (4.5 ms).
#include "mci_fast_group.hpp"

#include "mci_fast_dev.hpp"

#include <type_traits>

namespace mcid
{
namespace
{
// ---- within a group of L adjacent lanes ----
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true); }

template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = dpp<CTRL>((uint32_t)u), hi = dpp<CTRL>((uint32_t)(u >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

constexpr int quad(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }
constexpr int ROW_SHR1 = 0x111, ROW_HALF_MIRROR = 0x141;

// the value of the lane before; 0.0 in the group's first lane (keep: all ones elsewhere, 0 there)
template <int L>
__device__ __forceinline__ double from_prev(double v, uint32_t keep)
{
    constexpr int CTRL = L == 2 ? quad(0, 0, 2, 2) : L == 4 ? quad(0, 0, 1, 2) : ROW_SHR1;
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = dpp<CTRL>((uint32_t)u) & keep, hi = dpp<CTRL>((uint32_t)(u >> 32)) & keep;
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// the value of the group's last lane in every lane of the group
template <int L>
__device__ __forceinline__ double from_last(double v, int g)
{
    if constexpr (L == 2) { return dpp<quad(1, 1, 3, 3)>(v); }
    else if constexpr (L == 4) { return dpp<quad(3, 3, 3, 3)>(v); }
    else {
        const double q = dpp<quad(3, 3, 3, 3)>(v);    // the second quad holds it
        const double m = dpp<ROW_HALF_MIRROR>(q);     // and the first, mirrored
        return g < 4 ? m : q;
    }
}

// the value of the group's first lane in every lane of the group
template <int L>
__device__ __forceinline__ uint32_t from_first(uint32_t v, int g)
{
    if constexpr (L == 2) { return dpp<quad(0, 0, 2, 2)>(v); }
    else if constexpr (L == 4) { return dpp<quad(0, 0, 0, 0)>(v); }
    else {
        const uint32_t q = dpp<quad(0, 0, 0, 0)>(v);
        const uint32_t m = dpp<ROW_HALF_MIRROR>(q);
        return g < 4 ? q : m;
    }
}

// LDS written by one lane of the wave and read by another: the accesses of a wave are carried out in
// program order, so the compiler's order is all that has to hold
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// a 64-bit output of mt19937_64 in 32-bit halves: its shifts and masks are then single instructions
struct U64
{
    uint32_t lo, hi;
};
__device__ __forceinline__ U64 halves(uint64_t v) { return {(uint32_t)v, (uint32_t)(v >> 32)}; }
// the same word as a value of its own: a conversion of half of a 64-bit load is otherwise taken for
// one of the whole load shifted
__device__ __forceinline__ uint32_t apart(uint32_t v)
{
    asm("" : "+v"(v));
    return v;
}
__device__ __forceinline__ uint64_t whole(U64 v) { return ((uint64_t)v.hi << 32) | v.lo; }
// a ^ (b & c)
__device__ __forceinline__ uint32_t xor_and(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x78); }

// mt_twist of mci_device.hpp (of x[k + 1] only the low word counts)
__device__ __forceinline__ U64 mt_twist32(U64 xk, uint32_t xk1, U64 xkm)
{
    const uint32_t y = __builtin_amdgcn_bitop3_b32(xk.lo, xk1, 0x7fffffffu, 0xD8);  // the top bit of xk, the others of xk1
    const uint32_t odd = (uint32_t)((int32_t)(y << 31) >> 31);
    return {xor_and(xkm.lo ^ __builtin_amdgcn_alignbit(xk.hi, y, 1), odd, 0xa96619e9u),
            xor_and(xkm.hi ^ (xk.hi >> 1), odd, 0xb5026f5au)};
}

// mt_temper of mci_device.hpp
__device__ __forceinline__ U64 mt_temper32(U64 z)
{
    const uint32_t l1 = xor_and(z.lo, __builtin_amdgcn_alignbit(z.hi, z.lo, 29), 0x55555555u), h1 = xor_and(z.hi, z.hi >> 29, 5u);
    const uint32_t h2 = xor_and(h1, __builtin_amdgcn_alignbit(h1, l1, 15), 0x71d67fffu), l2 = xor_and(l1, l1 << 17, 0xeda60000u);
    const uint32_t h3 = xor_and(h2, l2 << 5, 0xfff7eee0u);
    return {l2 ^ (h3 >> 11), h3};
}

// uniform_real_distribution(-1, 1) on the canonical double of w: u = min(RN(w), the double below
// 2^64) 2^-64, then (u 2) + (-1).  Every scaling is exact, so each rounding is the reference's.
__device__ __forceinline__ double mt_symmetric(U64 w)
{
    const double v = fma((double)apart(w.hi), 0x1p32, (double)w.lo);
    return fma(fmin(v, 0x1.fffffffffffffp+63), 0x1p-63, -1.0);
}

// The generators of a wave's walkers in their groups' registers (groups of four lanes): element 4 i + g is
// register i of lane g, so that elements 156 apart share a lane.
constexpr int MT_NR = MT_N / 4;              // registers
constexpr int MT_RS = MT_NR / MT_SEG;        // registers of a part
constexpr int MT_RP = WAVE / 4 + 2;          // an LDS row: one output of each walker, padded so that a walker's
                                             // lanes reading rows some way apart use different banks
static_assert(MT_NR % MT_SEG == 0 && MT_N == MT_SEG * MT_CH && MT_N == 2 * MT_M && MT_M % 4 == 0, "");

// the state rotated so that its next index is 0 (the same generator)
__device__ __forceinline__ void mt_load(const FastArgs &A, int64_t w, int g, U64 (&m)[MT_NR])
{
    const int p0 = A.mtp[w];
#pragma unroll
    for (int i = 0; i < MT_NR; ++i) {
        const int k = i * 4 + g + p0;
        m[i] = halves(A.mt[(int64_t)(k < MT_N ? k : k - MT_N) * A.W + w]);
    }
}

// part q (a constant once unrolled) of a round: its elements by the lazy twist of mci_device.hpp's
// mt_next, their outputs to MT_CH rows from `row` (this walker's place in the first)
__device__ __forceinline__ void mt_part(U64 (&m)[MT_NR], int q, int g, uint64_t *row)
{
#pragma unroll
    for (int j = 0; j < MT_RS; ++j) {
        const int i = q * MT_RS + j;
        const uint32_t here = dpp<quad(1, 2, 3, 3)>(m[i].lo), next = dpp<quad(0, 0, 0, 0)>(m[(i + 1) % MT_NR].lo);
        m[i] = mt_twist32(m[i], g == 3 ? next : here, m[(i + MT_NR / 2) % MT_NR]);
        row[(j * 4 + g) * MT_RP] = whole(mt_temper32(m[i]));
    }
}

// The state back to memory, kt the next element of the round and `over` outputs made but not taken:
// their elements go back to their values before the twist, the last first.  new = far ^ (y >> 1) ^ (odd
// y ? A : 0) gives y (A's top bit is set), which holds the element's high 33 bits and the next element's
// low 31.
__device__ __forceinline__ void mt_store(const FastArgs &A, int64_t w, int g, const U64 (&m)[MT_NR], int kt, int over)
{
#pragma unroll
    for (int i = 0; i < MT_NR; ++i) { A.mt[(int64_t)(i * 4 + g) * A.W + w] = whole(m[i]); }
    __threadfence_block();
    auto at = [&](int k) -> uint64_t & { return A.mt[(int64_t)k * A.W + w]; };
    auto before = [&](int k) -> uint64_t {
        const uint64_t v = at(k) ^ at(k < MT_M ? k + MT_M : k - MT_M);
        const uint64_t odd = v >> 63;
        return ((v ^ (odd ? 0xb5026f5aa96619e9ULL : 0ULL)) << 1) | odd;
    };
    for (int r = 0; r < over; r += 4) {
        if (r + g < over) {
            int k = kt - 1 - r - g;
            if (k < 0) { k += MT_N; }
            const uint64_t y = before(k), yp = before(k > 0 ? k - 1 : MT_N - 1);
            at(k) = (y & 0xffffffff80000000ULL) | (yp & 0x7fffffffULL);
        }
    }
    if (g == 0) {
        const int k = kt - over;
        A.mtp[w] = k < 0 ? k + MT_N : k % MT_N;
    }
}

// Runs nsteps steps of `per` outputs each in the order of mt_parts (mci_fast_plan.hpp): step(row) takes them
// from consecutive rows (MT_RP apart) from `row`.
template <int LEFT, class F>
__device__ __forceinline__ void mt_run(const FastArgs &A, int64_t w, int g, uint64_t *mine, int per, F step)
{
    U64 m[MT_NR];
    mt_load(A, w, g, m);
    const MtEnd end = mt_parts<LEFT>(
        A.nsteps, per,
        [&](int from, int to, int n) {
            wave_order();
            if constexpr (LEFT == 4) {
                if (g < n) { mine[(to + g) * MT_RP] = mine[(from + g) * MT_RP]; }
            }
            else {
                for (int r = g; r < n; r += 4) { mine[(to + r) * MT_RP] = mine[(from + r) * MT_RP]; }
            }
        },
        [&](int q) {
            mt_part(m, q, g, mine + LEFT * MT_RP);
            wave_order();
        },
        [&](int row) { step(mine + row * MT_RP); });
    mt_store(A, w, g, m, end.next, end.over);
}

// q / div, the division (a dozen FP64 instructions) left out where it changes nothing: by 1, the default
__device__ __forceinline__ double over_div(double q, double div)
{
    if (div != 1.0) {
        asm volatile("");  // a branch, not a select of the finished division
        q = q / div;
    }
    return q;
}

// One walker on L lanes, S slots a lane.
//  Native streams (S even): a lane's slots are S consecutive main words of the step, so that its
//  Philox blocks are its own; word 0 is the acceptance word, word j coordinate j - 1.
//  Reference streams: a lane's slots are S consecutive coordinates.  EX: every slot holds one (d = L S).
template <int FL, int L, int S, bool EX>
__global__ __launch_bounds__(WAVE, (FL & F_MT) && S <= 4 ? 2 : 1) void k_fast64_grp(FastArgs A)
{
    constexpr bool FULL = (FL & F_FULL) != 0;
    constexpr bool HX2 = (FL & F_X2) != 0, HSUM = (FL & F_SUM) != 0, HEXP = (FL & F_EXP) != 0;
    constexpr bool ACC = (FL & 7) != 0 && !FULL;  // per-step block sums
    constexpr bool REC = HX2 && !FULL;             // per-coordinate block sums
    constexpr bool MT = (FL & F_MT) != 0;
    constexpr bool QN = HSUM || HEXP;              // |x|^2 is needed
    constexpr int WL = WAVE / L;                   // walkers of a wave
    extern __shared__ uint64_t st[];               // reference streams: outputs of the walkers' generators
    const int d = A.ndim;
    const int lane = threadIdx.x, g = lane & (L - 1), wl = lane / L;
    const int64_t W = A.W, B = A.blocksize;
    const int64_t w = (int64_t)blockIdx.x * WL + wl;
    const bool live = w < W && (!A.wcount || w < *A.wcount);
    double step = live ? A.steps[w] : 0.0;
    if (A.pend) {
        if (A.pend->apply && live) {
            step = step * A.pend->fact;
            for (int i = 0; i < d; ++i) {
                if (step > 0.5 * A.dimsizes[i]) { step = 0.5 * A.dimsizes[i]; }
            }
            if (step < (double)FLT_MIN) { step = (double)FLT_MIN; }
            if (g == 0) { A.steps[w] = step; }
        }
        if (A.pend->done) { return; }
    }
    if (!live || (A.active && !A.active[w])) { return; }
    const int c0 = g * S - (MT ? 0 : 1);  // the coordinate of slot 0
    double x[S], xn[S], sm[S], a[S];
    bool ok[S];                            // the slot holds a coordinate
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int c = c0 + s;
        ok[s] = EX || (c >= 0 && c < d);
        x[s] = 0.0;
        xn[s] = 0.0;
        sm[s] = 0.0;
        a[s] = 0.0;
        if (ok[s]) {
            x[s] = A.x64[(int64_t)c * W + w];
            a[s] = A.a ? A.a[c] : 1.0;
        }
    }
    const uint32_t keep = apart(g == 0 ? 0u : 0xFFFFFFFFu);
    // v_0 + v_1 + ... over the walker's coordinates in order, from 0.0 (empty slots hold 0.0): each
    // lane continues from the lane before, L times over, so that the last lane ends with the whole sum
    auto ordered = [&](const double (&v)[S]) __attribute__((always_inline)) -> double {
        double c = 0.0;
#pragma unroll
        for (int ph = 0; ph < L; ++ph) {
            if (ph > 0) { c = from_prev<L>(c, keep); }
#pragma unroll
            for (int s = 0; s < S; ++s) { c = c + v[s]; }
        }
        return from_last<L>(c, g);
    };
    double Sold, q = 0.0, e = 0.0, Sr = 0.0, Se = 0.0;
    {
        double p[S], p2[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            p2[s] = x[s] * x[s];
            p[s] = p2[s] * a[s];
        }
        Sold = ordered(p);
        if (QN) { q = ordered(p2); }
    }
    if (HEXP) { e = exp(-(q / A.exp_div)); }
    const uint32_t wid = A.wmap ? (uint32_t)A.wmap[w] : (uint32_t)w;
    [[maybe_unused]] uint64_t t = MT ? 0 : A.ctr[w];
    int64_t nacc = 0, inblk = 0, step_no = 0;
    // the next row of each observable's data, and this lane's place in a row in bytes (the host checks
    // that a row of x_i^2 is below 4 GiB): a uniform base and a 32-bit offset
    char *rx = reinterpret_cast<char *>(A.d_x2), *rs = reinterpret_cast<char *>(A.d_x2sum), *re = reinterpret_cast<char *>(A.d_exp);
    const int64_t w8 = W * 8, rowx = w8 * d;
    const uint32_t off = (uint32_t)w * 8u;
    uint32_t offx[S];
#pragma unroll
    for (int s = 0; s < S; ++s) { offx[s] = (uint32_t)((ok[s] ? c0 + s : 0) * w8) + off; }
    auto put = [](char *row, uint32_t o, double v) { *reinterpret_cast<double *>(row + o) = v; };

    // the step's proposal from the slots' random values r
    double p[S], p2[S];
    auto propose = [&](int s, double r) __attribute__((always_inline)) {
        double v = x[s] + step * r;
        if (!EX) { v = ok[s] ? v : 0.0; }
        xn[s] = v;
        p2[s] = v * v;
        p[s] = p2[s] * a[s];
    };
    // the decision from the acceptance word uw (native: the shared word; reference streams: the
    // acceptance output) and the observables after the step, as k_fast64_allr takes them
    // (inlined at each of its calls, whatever its size: a call of its own takes the walker's arrays by address,
    // and they then live in scratch memory)
    auto finish = [&](U64 uw) __attribute__((always_inline)) {
        const double Snew = ordered(p);
        double qn = 0.0;
        if (QN) { qn = ordered(p2); }
        const double ee = Sold - Snew;
        const float U = (float)apart(uw.hi);
        const float F = __builtin_amdgcn_exp2f(fmaf((float)ee, 0x1.715476p+0f, 32.0f));
        const float Facc = MT ? fmaf(F, 0.9999f, -3.0f) : fmaf(F, 0.9999f, -2.0f);
        const float Frej = MT ? fmaf(F, 1.0001f, 1.0f) : F * 1.0001f;
        bool acc = U < Facc;
        // (two ballots of plain compares: each is the compare's own lane mask)
        if (__builtin_expect((__builtin_amdgcn_ballot_w64(U <= Frej) & ~__builtin_amdgcn_ballot_w64(acc)) != 0, 0)) {
            const bool band = !acc && U <= Frej;
            double u;
            if (MT) { u = (mt_canonical(whole(uw)) * 1.0) + 0.0; }
            else {
                uint32_t l0, l1, l2, l3;
                philox(0x30000000u, wid, (uint32_t)t, (uint32_t)(t >> 32), A.key0, A.key1, l0, l1, l2, l3);
                u = (double)(whole({l0, uw.hi}) >> 11) * 0x1p-53;
            }
            if (band) { acc = u <= exp(ee); }
        }
        if (!MT) { ++t; }
        nacc += acc ? 1 : 0;
        Sold = acc ? Snew : Sold;
        if (QN) { q = acc ? qn : q; }
#pragma unroll
        for (int s = 0; s < S; ++s) { x[s] = acc ? xn[s] : x[s]; }
        if (HEXP && acc) { e = exp(-(q / A.exp_div)); }
        if (FULL) {
            if (HX2) {
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const double v = x[s] * x[s];
                    sm[s] = sm[s] + v;
                    if (ok[s]) { put(rx, offx[s], v); }
                }
                rx += rowx;
            }
            if (HSUM) {
                const double v = over_div(q, A.x2sum_div);
                Sr = Sr + v;
                if (g == 0) { put(rs, off, v); }
                rs += w8;
            }
            if (HEXP) {
                Se = Se + e;
                if (g == 0) { put(re, off, e); }
                re += w8;
            }
        }
        if (ACC) {
            if (REC) {
#pragma unroll
                for (int s = 0; s < S; ++s) { sm[s] = sm[s] + x[s] * x[s]; }
            }
            if (HSUM) { Sr = Sr + over_div(q, A.x2sum_div); }
            if (HEXP) { Se = Se + e; }
            if (++inblk == B) {
                const double norm = 1. / (double)B;
                if (REC) {
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        if (ok[s]) { put(rx, offx[s], sm[s] * norm); }
                        sm[s] = 0.0;
                    }
                    rx += rowx;
                }
                if (HSUM) {
                    if (g == 0) { put(rs, off, Sr * norm); }
                    rs += w8;
                }
                if (HEXP) {
                    if (g == 0) { put(re, off, Se * norm); }
                    re += w8;
                }
                Sr = 0.0;
                Se = 0.0;
                inblk = 0;
            }
        }
        ++step_no;
    };

    if constexpr (MT) {
        static_assert(L == 4, "the generator's elements lie on four lanes");
        mt_run<L * S>(A, w, g, st + wl, d + 1, [&](const uint64_t *row) {
            U64 o[S];
            const U64 uo = halves(row[d * MT_RP]);
#pragma unroll
            for (int s = 0; s < S; ++s) { o[s] = halves(row[(g * S + s) * MT_RP]); }
#pragma unroll
            for (int s = 0; s < S; ++s) { propose(s, mt_symmetric(o[s])); }
            finish(uo);
        });
    }
    else {
        constexpr int NB = S / 2;  // the lane's Philox blocks of a step pair
        auto rnd = [](uint32_t v) { return fma((double)v, 0x1p-31, -(1.0 - 0x1p-32)); };
        uint32_t sw[S];  // the second step's words of a pair
        auto single = [&]() __attribute__((always_inline)) {
            const uint32_t par = (uint32_t)(t & 1u);
            const uint64_t tp = t >> 1;
            uint32_t uw = 0;
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                uint32_t o0, o1, o2, o3;
                philox((uint32_t)(g * NB + k), wid, (uint32_t)tp, (uint32_t)(tp >> 32), A.key0, A.key1, o0, o1, o2, o3);
                const uint32_t wa = par ? o2 : o0, wb = par ? o3 : o1;
                if (k == 0) { uw = wa; }
                propose(2 * k, rnd(wa));
                propose(2 * k + 1, rnd(wb));
            }
            finish({0u, from_first<L>(uw, g)});
        };
        // lanes whose counters differ in parity (a restored state can set them so) step alone
        const uint64_t podd = __builtin_amdgcn_ballot_w64((t & 1u) != 0);
        const bool pairs = podd == 0 || podd == __builtin_amdgcn_ballot_w64(true);
        if (pairs) {
            if ((t & 1u) && step_no < A.nsteps) { single(); }
            while (step_no + 2 <= A.nsteps) {
                const uint64_t tp = t >> 1;
                uint32_t uw = 0;
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    uint32_t o0, o1, o2, o3;
                    philox((uint32_t)(g * NB + k), wid, (uint32_t)tp, (uint32_t)(tp >> 32), A.key0, A.key1, o0, o1, o2, o3);
                    sw[2 * k] = o2;
                    sw[2 * k + 1] = o3;
                    if (k == 0) { uw = o0; }
                    propose(2 * k, rnd(o0));
                    propose(2 * k + 1, rnd(o1));
                }
                finish({0u, from_first<L>(uw, g)});
#pragma unroll
                for (int s = 0; s < S; ++s) { propose(s, rnd(sw[s])); }
                finish({0u, from_first<L>(sw[0], g)});
            }
        }
        while (step_no < A.nsteps) { single(); }
        if (g == 0) { A.ctr[w] = t; }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (ok[s]) {
            A.x64[(int64_t)(c0 + s) * W + w] = x[s];
            if (FULL && HX2 && A.s_x2) { A.s_x2[(int64_t)(c0 + s) * W + w] = sm[s]; }
        }
    }
    if (g == 0) {
        if (FULL && HSUM && A.s_x2sum) { A.s_x2sum[w] = Sr; }
        if (FULL && HEXP && A.s_exp) { A.s_exp[w] = Se; }
        A.acc[w] = nacc;
        A.rej[w] = A.nsteps - nacc;
    }
}

// Single-coordinate moves (SRRDVecMove, veclen 1, one step size) on the reference streams, a walker on
// four lanes of S coordinates each (d = 2^m: 4 S, or fewer with S = 1).  A step takes three outputs: the
// coordinate (the top m bits), the proposal and the acceptance uniform; the lane that owns the coordinate
// decides, with k_fast64's screen and arithmetic, and every lane adds its coordinates' values to their
// per-step sums, so every number is bit-identical to the generic kernel.
//
// On one lane a walker (k_fast64) the sums read and wrote the walker's 16-byte records in LDS every step
// and the outputs moved 72 bytes of generator state in HBM: 14.3 ms for 65,536 walkers x 10,240 steps at
// d = 16 (48.9 GB at 3.4 TB/s).  Here both stay in registers: 8.9 ms, bound by instruction issue.
template <int FL, int S>
__global__ __launch_bounds__(WAVE, S <= 4 ? 2 : 1) void k_fast64_vec4(FastArgs A)
{
    constexpr bool FULL = (FL & F_FULL) != 0;
    constexpr bool HX2 = (FL & F_X2) != 0, HSUM = (FL & F_SUM) != 0, HEXP = (FL & F_EXP) != 0;
    constexpr bool ACC = (FL & 7) != 0 && !FULL, QN = HSUM || HEXP;
    constexpr int L = 4, WL = WAVE / L;
    extern __shared__ uint64_t st[];
    const int d = A.ndim;
    const int lane = threadIdx.x, g = lane & (L - 1), wl = lane / L;
    const int64_t W = A.W, B = A.blocksize;
    const int64_t w = (int64_t)blockIdx.x * WL + wl;
    const bool live = w < W && (!A.wcount || w < *A.wcount);
    double step = live ? A.steps[w] : 0.0;
    if (A.pend) {
        if (A.pend->apply && live) {
            step = step * A.pend->fact;
            for (int i = 0; i < d; ++i) {
                if (step > 0.5 * A.dimsizes[i]) { step = 0.5 * A.dimsizes[i]; }
            }
            if (step < (double)FLT_MIN) { step = (double)FLT_MIN; }
            if (g == 0) { A.steps[w] = step; }
        }
        if (A.pend->done) { return; }
    }
    if (!live || (A.active && !A.active[w])) { return; }
    const int c0 = g * S;
    const bool mine = c0 < d;  // a lane holds S coordinates or (d < 4) none
    double x[S], q2[S], sm[S];
    float cs[S];               // the screen's -a_i log2 e
    uint32_t offx[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        x[s] = 0.0;
        sm[s] = 0.0;
        cs[s] = 0.0f;
        if (mine) {
            x[s] = A.x64[(int64_t)(c0 + s) * W + w];
            cs[s] = (float)(-A.a[c0 + s] * 0x1.71547652b82fep+0);
        }
        q2[s] = x[s] * x[s];
        offx[s] = (uint32_t)((mine ? c0 + s : 0) * W * 8) + (uint32_t)w * 8u;
    }
    const uint32_t keep = apart(g == 0 ? 0u : 0xFFFFFFFFu);
    auto ordered = [&](const double (&v)[S]) __attribute__((always_inline)) -> double {  // as in k_fast64_grp
        double c = 0.0;
#pragma unroll
        for (int ph = 0; ph < L; ++ph) {
            if (ph > 0) { c = from_prev<L>(c, keep); }
#pragma unroll
            for (int s = 0; s < S; ++s) { c = c + v[s]; }
        }
        return from_last<L>(c, g);
    };
    double e = 0.0, Sr = 0.0, Se = 0.0;
    if (HEXP) { e = exp(-(ordered(q2) / A.exp_div)); }
    int64_t nacc = 0, inblk = 0;
    char *rx = reinterpret_cast<char *>(A.d_x2), *rs = reinterpret_cast<char *>(A.d_x2sum), *re = reinterpret_cast<char *>(A.d_exp);
    const int64_t w8 = W * 8, rowx = w8 * d;
    const uint32_t off = (uint32_t)w * 8u;
    auto put = [](char *row, uint32_t o, double v) { *reinterpret_cast<double *>(row + o) = v; };
    const uint32_t ibits = (uint32_t)A.ibits, vshift = (uint32_t)A.vshift;
    mt_run<4>(A, w, g, st + wl, 3, [&](const uint64_t *row) {
        const U64 oi = halves(row[0]), op = halves(row[MT_RP]), uw = halves(row[2 * MT_RP]);
        const uint32_t v = __builtin_amdgcn_ubfe(apart(oi.hi), vshift, ibits);
        const int slot = (int)(v & (S - 1));
        const bool own = v / S == (uint32_t)g;
        double xo = x[0];
        float cv = cs[0];
#pragma unroll
        for (int s = 1; s < S; ++s) {
            xo = slot == s ? x[s] : xo;
            cv = slot == s ? cs[s] : cv;
        }
        const double xn = xo + step * mt_symmetric(op);
        const double xn2 = xn * xn, xo2 = xo * xo;
        const float U = (float)apart(uw.hi);
        const float F = __builtin_amdgcn_exp2f(fmaf((float)(xn2 - xo2), cv, 32.0f));
        const float Facc = fmaf(F, 0.9999f, -3.0f), Frej = fmaf(F, 1.0001f, 1.0f);
        bool acc = U < Facc;
        if (__builtin_expect((__builtin_amdgcn_ballot_w64(U <= Frej) & ~__builtin_amdgcn_ballot_w64(acc) & __builtin_amdgcn_ballot_w64(own)) != 0, 0)) {
            if (own && !acc && U <= Frej) {
                const double av = A.a[v];
                const double ex = xn2 * av - xo2 * av;
                acc = (mt_canonical(whole(uw)) * 1.0) + 0.0 <= exp(-ex);
            }
        }
        acc = acc && own;
        nacc += acc ? 1 : 0;
        const int to = acc ? slot : -1;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            x[s] = to == s ? xn : x[s];
            q2[s] = to == s ? xn2 : q2[s];
        }
        if (!(ACC || FULL)) { return; }
        double q = 0.0;
        if (QN) { q = ordered(q2); }
        if (HEXP) {
            uint32_t any = acc ? 1u : 0u;  // some lane of the group moved
            any |= dpp<quad(1, 0, 3, 2)>(any);
            any |= dpp<quad(2, 3, 0, 1)>(any);
            if (any) { e = exp(-(q / A.exp_div)); }
        }
        if (HX2) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                sm[s] = sm[s] + q2[s];
                if (FULL && mine) { put(rx, offx[s], q2[s]); }
            }
            if (FULL) { rx += rowx; }
        }
        if (HSUM) {
            const double t = over_div(q, A.x2sum_div);
            Sr = Sr + t;
            if (FULL) {
                if (g == 0) { put(rs, off, t); }
                rs += w8;
            }
        }
        if (HEXP) {
            Se = Se + e;
            if (FULL) {
                if (g == 0) { put(re, off, e); }
                re += w8;
            }
        }
        if (ACC && ++inblk == B) {
            const double norm = 1. / (double)B;
            if (HX2) {
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    if (mine) { put(rx, offx[s], sm[s] * norm); }
                    sm[s] = 0.0;
                }
                rx += rowx;
            }
            if (HSUM) {
                if (g == 0) { put(rs, off, Sr * norm); }
                rs += w8;
            }
            if (HEXP) {
                if (g == 0) { put(re, off, Se * norm); }
                re += w8;
            }
            Sr = 0.0;
            Se = 0.0;
            inblk = 0;
        }
    });
    // the walker's accepted steps: the sum over its lanes
    auto plus = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const uint64_t u = (uint64_t)nacc;
        nacc += (int64_t)(((uint64_t)dpp<C>((uint32_t)(u >> 32)) << 32) | dpp<C>((uint32_t)u));
    };
    plus(std::integral_constant<int, quad(1, 0, 3, 2)>{});
    plus(std::integral_constant<int, quad(2, 3, 0, 1)>{});
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (mine) {
            A.x64[(int64_t)(c0 + s) * W + w] = x[s];
            if (FULL && HX2 && A.s_x2) { A.s_x2[(int64_t)(c0 + s) * W + w] = sm[s]; }
        }
    }
    if (g == 0) {
        if (FULL && HSUM && A.s_x2sum) { A.s_x2sum[w] = Sr; }
        if (FULL && HEXP && A.s_exp) { A.s_exp[w] = Se; }
        A.acc[w] = nacc;
        A.rej[w] = A.nsteps - nacc;
    }
}

template <int FL>
bool go_vec(int S, hipStream_t s, const FastArgs &A)
{
    const size_t sh = sizeof(uint64_t) * (4 + MT_CH) * MT_RP;
    const dim3 grid((unsigned)((A.W + WAVE / 4 - 1) / (WAVE / 4)));
    switch (S) {
#define SLOTS(n)                                                                                         \
    case n: hipLaunchKernelGGL((k_fast64_vec4<FL, n>), grid, dim3(WAVE), sh, s, A); return true;
        SLOTS(1) SLOTS(2) SLOTS(4) SLOTS(8) SLOTS(16)
#undef SLOTS
    }
    return false;
}

template <int FL, int L, int S>
void go(hipStream_t s, const FastArgs &A)
{
    constexpr int WL = WAVE / L;
    constexpr bool MT = (FL & F_MT) != 0;
    const size_t sh = MT ? sizeof(uint64_t) * (L * S + MT_CH) * MT_RP : 0;
    const dim3 grid((unsigned)((A.W + WL - 1) / WL));
    if constexpr (MT && (S & (S - 1)) == 0) {
        if (A.ndim == L * S) {
            hipLaunchKernelGGL((k_fast64_grp<FL, L, S, true>), grid, dim3(WAVE), sh, s, A);
            return;
        }
    }
    hipLaunchKernelGGL((k_fast64_grp<FL, L, S, false>), grid, dim3(WAVE), sh, s, A);
}

template <int FL>
bool go_shape(int L, int S, hipStream_t s, const FastArgs &A)
{
#define SHAPE(l, n)                                                                                      \
    if (L == l && S == n) {                                                                              \
        go<FL, l, n>(s, A);                                                                              \
        return true;                                                                                     \
    }
    if constexpr ((FL & F_MT) != 0) { GROUP_SHAPES_MT(SHAPE) }
    else { GROUP_SHAPES(SHAPE) }
#undef SHAPE
    return false;
}
} // namespace

// this file is compiled once for each part of the forms (the build defines GROUP_PART)
#define GROUP_NAME2(n) launch_group_##n
#define GROUP_NAME(n) GROUP_NAME2(n)
bool GROUP_NAME(GROUP_PART)(int fl, bool vec, int L, int S, const FastArgs &A, hipStream_t s)
{
    switch (fl) {
#define FORM(f)                                                                                          \
    case f: return !vec && go_shape<f>(L, S, s, A);                                                     \
    case f + F_MT: return vec ? go_vec<f + F_MT>(S, s, A) : go_shape<f + F_MT>(L, S, s, A);
#if GROUP_PART == 0
        FORM(0) FORM(1)
#elif GROUP_PART == 1
        FORM(2) FORM(3)
#elif GROUP_PART == 2
        FORM(4) FORM(5)
#elif GROUP_PART == 3
        FORM(6) FORM(7)
#elif GROUP_PART == 4
        FORM(17) FORM(18)
#elif GROUP_PART == 5
        FORM(19) FORM(20)
#elif GROUP_PART == 6
        FORM(21) FORM(22) FORM(23)
#endif
#undef FORM
    }
    return false;
}
} // namespace mcid
