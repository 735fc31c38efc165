// mci_mlp_step.hip — a training iteration in three kernels.
//
// k_step_tile: one workgroup of 16 waves takes 16 samples through the whole network and back.  The
// samples' activations stay in LDS (pre-activations in FP32, the products' operands in BF16), the
// weights come from the L2 in operand order: at the learned proposal's size (d 32, H 128, 576 outputs) 375 KB per
// workgroup, 96 MB for the 256 workgroups of 4096 samples.  Every product is
// v_mfma_f32_16x16x32_bf16 with the features as rows and the samples as columns: lane l supplies row or
// column l % 16 and terms 8 (l / 16) .. + 7 of the reduction, accumulator element i of lane l is
// C[4 (l / 16) + i][l % 16] (the layouts were checked on the device).  A wave owns the same feature
// tiles forward and backward, so a pre-activation is read back by the lane that wrote it.
//
// k_step_wgrad: the weight gradients dW[a][b] = sum over samples A[a][s] B[b][s] from the tiles'
// BF16 arrays [tile][feature][16], in which a lane's operand of v_mfma_f32_32x32x16_bf16 is 16
// contiguous bytes and a wave's a contiguous KB: no LDS staging, no transposes.  A workgroup's eight
// waves share the samples of one 32 x 32 tile and add up in LDS.  The bias gradients' sums over the
// sample tiles are workgroups of the same launch.
//
// k_step_adam: splits added in their order, Adam, and the BF16 copies in the forms the next iteration
// reads.
//
// What bounds it: latency.  4096 samples are one workgroup per compute unit, and a layer is one or two
// round trips to the L2 and a barrier.  Measured at d 32, H 128, K 8 and 4096 samples: 24.7 + 8.3 + 5.1 us
// an iteration (tile, weight gradients, Adam), 42 us with the launches; as separate products, row sums and
// elementwise passes (about 25 launches, 50 MB of activations through memory) 276 us.  With row-major
// weights (half lines per request), no warming of the L2, 64-bit remainders in the pairs and one wave per
// tile of the backward products the tile took 35.6 us.  Tiles past the LDS of a compute unit (d > 75 at
// H 128, K 8; H > 512 at d 32) train by separate products.
#include "mci_mlp_step.hpp"

namespace mcim
{
namespace
{
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int NS = STEP_NS;
constexpr int TPB = 1024, NWAVE = TPB / 64; // k_step_tile
constexpr int PAD = 8;                      // BF16 operand rows in LDS: a multiple of 16 bytes that walks over the banks
constexpr int WTPB = 512, WWAVE = WTPB / 64; // k_step_wgrad

__device__ __forceinline__ bf16_t f2bf(float f)
{
    // round to nearest even (finite inputs)
    const uint32_t u = __float_as_uint(f);
    return (bf16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ bf16x8 load8(const bf16_t *p) { return *reinterpret_cast<const bf16x8 *>(p); }

__device__ __forceinline__ void philox(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1, uint32_t o[4])
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r > 0) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    o[0] = c0; o[1] = c1; o[2] = c2; o[3] = c3;
}

// C[16 ft .. + 15][sample] for the wave's feature tiles ft: Wt [16 ntiles][kp] in operand order, xs
// [NS][kp + PAD] in LDS, kp a multiple of 32.  Eight loads are in flight at once (the last group's surplus
// ones repeat the last term's address and are not used).  Where the tiles leave half of the waves idle and
// `half` is given, waves ft and ft + 8 take half of the reduction each and add up there.
template <class F>
__device__ __forceinline__ void layer(const bf16_t *__restrict__ Wt, int ntiles, int kp, const bf16_t *xs, float *half, F epilogue)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nk = kp / 32;
    const bf16_t *b = xs + (lane & 15) * (kp + PAD) + 8 * (lane >> 4);
    const bool two = half && ntiles <= NWAVE / 2;
    const int kb = two && wave >= NWAVE / 2 ? nk / 2 : 0, ke = two && wave < NWAVE / 2 ? nk / 2 : nk;
    f32x4 acc = {};
    for (int ft = two ? wave & (NWAVE / 2 - 1) : wave; ft < ntiles; ft += NWAVE) {
        const bf16_t *a = Wt + (int64_t)ft * nk * 512 + lane * 8;
        acc = {};
        for (int k = kb; k < ke; k += 8) {
            bf16x8 av[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) { av[q] = load8(a + 512 * min(k + q, nk - 1)); }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (k + q < ke) { acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[q], load8(b + 32 * (k + q)), acc, 0, 0, 0); }
            }
        }
        if (!two) { epilogue(ft * 16 + 4 * (lane >> 4), lane & 15, acc); }
    }
    if (two) { // (the same for the whole workgroup)
        f32x4 *h = reinterpret_cast<f32x4 *>(half) + (wave & (NWAVE / 2 - 1)) * 64 + lane;
        if (wave >= NWAVE / 2) { *h = acc; }
        __syncthreads();
        if (wave < ntiles) { epilogue(wave * 16 + 4 * (lane >> 4), lane & 15, acc + *h); }
    }
}

__device__ __forceinline__ float sum16(float v) // over the 16 samples of a lane's quarter
{
    v += __shfl_xor(v, 1);
    v += __shfl_xor(v, 2);
    v += __shfl_xor(v, 4);
    return v + __shfl_xor(v, 8);
}

struct Lds
{
    float *z1, *z2, *out, *y, *part, *half;
    bf16_t *x, *h1, *h2, *dout;
};

// the tile's LDS: pointers into base, or (SIZE) only its length
template <bool SIZE>
__host__ __device__ inline size_t lds_layout(int d, int dp, int Hp, int Op, char *base, Lds &L)
{
    size_t o = 0;
    auto take = [&](size_t bytes) {
        char *p = SIZE ? nullptr : base + o;
        o += (bytes + 15) & ~(size_t)15;
        return p;
    };
    L.z1 = (float *)take(sizeof(float) * Hp * NS);
    L.z2 = (float *)take(sizeof(float) * Hp * NS);
    L.out = (float *)take(sizeof(float) * Op * NS);
    L.y = (float *)take(sizeof(float) * d * NS);
    L.part = (float *)take(sizeof(float) * 2 * 8 * NS);
    L.half = (float *)take(Hp <= 8 * NWAVE ? sizeof(f32x4) * 64 * (NWAVE / 2) : 0);
    L.x = (bf16_t *)take(sizeof(bf16_t) * NS * (dp + PAD));
    L.h1 = (bf16_t *)take(sizeof(bf16_t) * NS * (Hp + PAD));
    L.h2 = (bf16_t *)take(sizeof(bf16_t) * NS * (Hp + PAD));
    L.dout = (bf16_t *)take(sizeof(bf16_t) * NS * (Op + PAD));
    return o;
}

__global__ __launch_bounds__(TPB) void k_step_tile(StepNet N, StepBatch B, StepWork w, float inv_n)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    Lds L;
    const int d = N.d, H = N.H, K = N.K, Op = N.Op, dp = N.dp, Hp = N.Hp;
    lds_layout<false>(d, dp, Hp, Op, smem, L);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t tile = blockIdx.x;
    const int s = tid & 15;
    const int64_t r = tile * NS + s;
    const bool ok = r < B.n;
    float *bias = w.bias + tile * (Op + 2 * Hp);

    // the samples; meanwhile an XCD's workgroups bring the weights, which the last update left in other
    // XCDs' caches and in memory, into its L2, a slice each (blocks go round the eight XCDs)
    const int slices = max(1, min(32, (int)(gridDim.x / 8))), line = (int)(blockIdx.x / 8) % slices + slices * tid;
    uint32_t warm = 0;
    if (line < N.lines) { warm = *reinterpret_cast<const uint32_t *>(N.W1t + (int64_t)line * 64); }
    {
        int64_t at = r, bt = r, sa = B.n, sb = B.n;
        const float *a = B.X, *b = B.Y;
        if (B.snap) {
            uint32_t o[4];
            philox(0x30000000u, (uint32_t)r, (uint32_t)B.iter, (uint32_t)(B.iter >> 32), B.k0, B.k1, o);
            const int s1 = (int)(o[0] % (uint32_t)B.nsnap);
            int s2 = (int)(o[2] % (uint32_t)B.nsnap);
            const uint32_t W = (uint32_t)B.W; // <= 2^30
            at = (int64_t)(o[1] % W);
            const bool same = (float)(o[3] >> 24) * 0x1p-8f < B.same_frac;
            bt = same ? at : (int64_t)((o[3] & 0xffffffu) % W);
            if (same && B.nsnap > 1 && s2 == s1) { s2 = (s1 + 1) % B.nsnap; }
            a = B.snap + (int64_t)s1 * d * B.W;
            b = B.snap + (int64_t)s2 * d * B.W;
            sa = sb = B.W;
        }
        bf16_t *X = w.X + tile * dp * NS;
        for (int j = tid >> 4; j < dp; j += TPB / NS) {
            float xv = 0.f, yv = 0.f;
            if (ok && j < d) {
                xv = B.fixed_ctx ? B.fixed_ctx[j] : a[j * sa + at];
                yv = b[j * sb + bt];
            }
            const bf16_t xb = f2bf(xv * IN_SCALE);
            L.x[s * (dp + PAD) + j] = xb;
            X[j * NS + s] = xb;
            if (j < d) { L.y[j * NS + s] = yv; }
        }
    }
    asm volatile("" ::"v"(warm));
    __syncthreads();

    // forward: z = W h + b, h = silu(z)
    auto hidden = [&](float *z, bf16_t *h, bf16_t *hg, int64_t ob) {
        hg += tile * Hp * NS;
        return [=](int f, int c, f32x4 acc) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = acc[i] + (f + i < H ? N.p[ob + f + i] : 0.f);
                const bf16_t hv = f2bf(v / (1.0f + __expf(-v)));
                z[(f + i) * NS + c] = v;
                h[c * (Hp + PAD) + f + i] = hv;
                hg[(f + i) * NS + c] = hv;
            }
        };
    };
    layer(N.W1t, Hp / 16, dp, L.x, nullptr, hidden(L.z1, L.h1, w.H1, N.ob1));
    __syncthreads();
    layer(N.W2t, Hp / 16, Hp, L.h1, nullptr, hidden(L.z2, L.h2, w.H2, N.ob2));
    __syncthreads();
    layer(N.W3t, Op / 16, Hp, L.h2, nullptr, [&](int f, int c, f32x4 acc) {
#pragma unroll
        for (int i = 0; i < 4; ++i) { L.out[(f + i) * NS + c] = acc[i] + N.p[N.ob3 + f + i]; }
    });
    __syncthreads();

    // the head: waves k and k + 8 take component k, a lane one sample and every eighth coordinate.  The
    // softmax over the components is computed by every thread for its sample.
    {
        constexpr float HALF_LOG_2PI = 0.91893853320467274f;
        const int k = wave & 7, j0 = (wave >> 3) * 4 + (lane >> 4);
        const int L0 = 2 * d * K; // first logit row
        float a[8], amax = -__builtin_huge_valf(), asum = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            a[q] = q < K ? L.out[(L0 + q) * NS + s] : -__builtin_huge_valf();
            amax = fmaxf(amax, a[q]);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) { asum += q < K ? __expf(a[q] - amax) : 0.f; }
        const float lsa = amax + __logf(asum);
        float c = 0.f;
        if (k < K) {
            for (int j = j0; j < d; j += 8) {
                const float mu = MU_SCALE * L.out[(2 * d * k + j) * NS + s];
                const float ls = fminf(fmaxf(L.out[(2 * d * k + d + j) * NS + s], -LS_MAX), LS_MAX);
                const float z = (L.y[j * NS + s] - mu) * __expf(-ls);
                c += -ls - HALF_LOG_2PI - 0.5f * z * z;
            }
        }
        c += __shfl_xor(c, 16);
        c += __shfl_xor(c, 32);
        if (lane < NS) { L.part[wave * NS + s] = c; }
        __syncthreads();
        float cmax = -__builtin_huge_valf(), csum = 0.f, ck = 0.f, ak = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            // a[q] becomes component q's log-density
            const float al = a[q] - lsa;
            a[q] = q < K ? al + (L.part[q * NS + s] + L.part[(q + 8) * NS + s]) : -__builtin_huge_valf();
            cmax = fmaxf(cmax, a[q]);
            if (q == k) { ck = a[q]; ak = al; }
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) { csum += q < K ? __expf(a[q] - cmax) : 0.f; }
        const float lq = cmax + __logf(csum);
        bf16_t *dO = w.dO + tile * Op * NS;
        bf16_t *ds = L.dout + s * (Op + PAD);
        auto put = [&](int row, float g) {
            const float v = ok ? g : 0.f;
            const bf16_t vb = f2bf(v);
            L.out[row * NS + s] = v;
            ds[row] = vb;
            dO[row * NS + s] = vb;
        };
        if (k < K) {
            const float gam = __expf(ck - lq);
            if (tid < NS && ok) { w.loss[r] = -lq; }
            if (j0 == 0) { put(L0 + k, inv_n * (__expf(ak) - gam)); }
            for (int j = j0; j < d; j += 8) {
                const int im = 2 * d * k + j, il = im + d;
                const float mu = MU_SCALE * L.out[im * NS + s];
                const float ol = L.out[il * NS + s];
                const float ls = fminf(fmaxf(ol, -LS_MAX), LS_MAX);
                const float isg = __expf(-ls);
                const float z = (L.y[j * NS + s] - mu) * isg;
                put(im, inv_n * (-gam * z * isg) * MU_SCALE);
                put(il, fabsf(ol) < LS_MAX ? inv_n * gam * (1.0f - z * z) : 0.0f);
            }
        }
        for (int row = K * (1 + 2 * d) + (tid >> 4); row < Op; row += TPB / NS) { put(row, 0.f); }
    }
    __syncthreads();
    for (int f = tid; f < Op; f += TPB) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < NS; ++i) { v += L.out[f * NS + ((i + f) & (NS - 1))]; } // (each lane from its own bank)
        bias[f] = v;
    }

    // backward: dz = (W dz') silu'(z); its operand copy overwrites the activations no longer needed
    auto back = [&](const float *z, bf16_t *h, bf16_t *dg, float *bg) {
        dg += tile * Hp * NS;
        return [=](int f, int c, f32x4 acc) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float zz = z[(f + i) * NS + c];
                const float sg = 1.0f / (1.0f + __expf(-zz));
                const float v = acc[i] * (sg * (1.0f + zz * (1.0f - sg)));
                const bf16_t vb = f2bf(v);
                if (h) { h[c * (Hp + PAD) + f + i] = vb; }
                dg[(f + i) * NS + c] = vb;
                const float sum = sum16(v);
                if (c == 0) { bg[f + i] = sum; }
            }
        };
    };
    layer(N.W3, Hp / 16, Op, L.dout, L.half, back(L.z2, L.h2, w.dZ2, bias + Op));
    __syncthreads();
    layer(N.W2, Hp / 16, Hp, L.h2, nullptr, back(L.z1, nullptr, w.dZ1, bias + Op + Hp));
}

// one weight matrix: A, B as [tile][rows][16]; its gradient [na][nb] at off, row stride nb
struct WJob
{
    const bf16_t *A, *B;
    int ra, rb, na, nb;
    int64_t off;
};

__global__ __launch_bounds__(WTPB) void k_step_wgrad(WJob j1, WJob j2, WJob j3, StepNet N, const float *bias, float *ws, int64_t tiles)
{
    __shared__ float red[WWAVE][16][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int z = blockIdx.y, S = gridDim.y;
    const int64_t t0 = tiles * z / S, t1 = tiles * (z + 1) / S;
    ws += (int64_t)z * N.npad;
    int b = blockIdx.x;
    const int n1 = (j1.ra / 32) * (j1.rb / 32), n2 = (j2.ra / 32) * (j2.rb / 32), n3 = (j3.ra / 32) * (j3.rb / 32);
    if (b >= n1 + n2 + n3) { // biases: 64 of [b3 | b2 | b1], a wave every eighth tile
        const int PB = N.Op + 2 * N.Hp;
        const int f = (b - n1 - n2 - n3) * 64 + lane;
        float v = 0.f;
        if (f < PB) {
#pragma unroll 4
            for (int64_t t = t0 + wave; t < t1; t += WWAVE) { v += bias[t * PB + f]; }
        }
        red[wave][0][lane] = v;
        __syncthreads();
        if (wave == 0 && f < PB) {
            float g = 0.f;
            for (int q = 0; q < WWAVE; ++q) { g += red[q][0][lane]; }
            if (f < N.Op) { ws[N.ob3 + f] = g; }
            else if (f < N.Op + N.Hp) {
                if (f - N.Op < N.H) { ws[N.ob2 + f - N.Op] = g; }
            }
            else if (f - N.Op - N.Hp < N.H) { ws[N.ob1 + f - N.Op - N.Hp] = g; }
        }
        return;
    }
    WJob J = j3;
    if (b < n3) {}
    else if (b < n3 + n2) { J = j2; b -= n3; }
    else { J = j1; b -= n3 + n2; }
    const int cb = J.rb / 32, a0 = (b / cb) * 32, b0 = (b % cb) * 32;
    const bf16_t *A = J.A + (a0 + (lane & 31)) * NS + 8 * (lane >> 5);
    const bf16_t *Bp = J.B + (b0 + (lane & 31)) * NS + 8 * (lane >> 5);
    const int64_t sa = (int64_t)J.ra * NS, sb = (int64_t)J.rb * NS;
    f32x16 acc = {};
#pragma unroll 4
    for (int64_t t = t0 + wave; t < t1; t += WWAVE) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(load8(A + t * sa), load8(Bp + t * sb), acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) { red[wave][i][lane] = acc[i]; }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 1024 / WTPB; ++q) {
        const int i = (tid >> 6) + q * WWAVE;
        float v = 0.f;
#pragma unroll
        for (int u = 0; u < WWAVE; ++u) { v += red[u][i][lane]; }
        const int row = a0 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3), col = b0 + (lane & 31);
        if (row < J.na && col < J.nb) { ws[J.off + (int64_t)row * J.nb + col] = v; }
    }
}

// parameter i's BF16 value into the copies
__device__ __forceinline__ void put_copies(const StepNet &N, int64_t i, bf16_t v)
{
    const int H = N.H, Op = N.Op;
    if (i >= N.oW3) {
        if (i >= N.ob3) { return; }
        const int e = (int)(i - N.oW3), h = e / Op, o = e % Op;
        N.W3[step_operand(h, o, Op)] = v;
        N.W3t[step_operand(o, h, N.Hp)] = v;
    }
    else if (i >= N.oW2) {
        if (i >= N.ob2) { return; }
        const int e = (int)(i - N.oW2), k = e / H, f = e % H;
        N.W2[step_operand(k, f, N.Hp)] = v;
        N.W2t[step_operand(f, k, N.Hp)] = v;
    }
    else if (i < N.ob1) {
        const int e = (int)i, k = e / H, f = e % H;
        N.W1t[step_operand(f, k, N.dp)] = v;
    }
}

__global__ void k_step_copies(StepNet N)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N.npad) { put_copies(N, i, f2bf(N.p[i])); }
}

template <bool ADAM>
__global__ void k_step_adam(StepNet N, const float *ws, int S, float *g, float *p, float *m, float *v, bf16_t *pb, float lr, float b1,
                            float b2, float eps, float bc1, float bc2)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N.npad) { return; }
    float gi = 0.f;
#pragma unroll 4
    for (int z = 0; z < S; ++z) { gi += ws[(int64_t)z * N.npad + i]; }
    g[i] = gi;
    if (!ADAM) { return; }
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
    p[i] = pi;
    const bf16_t c = f2bf(pi);
    pb[i] = c;
    put_copies(N, i, c);
}

int64_t tiles_of(int64_t n) { return (n + NS - 1) / NS; }

int wgrad_tiles(const StepNet &N) { return (N.dp / 32 + N.Hp / 32 + N.Op / 32) * (N.Hp / 32); }
} // namespace

size_t step_lds(int d, int H, int Op)
{
    Lds L;
    return lds_layout<true>(d, (d + 31) / 32 * 32, (H + 31) / 32 * 32, Op, nullptr, L);
}

// enough workgroups to fill the chip twice, while each of a workgroup's eight waves keeps two sample
// tiles or more
int step_splits(const StepNet &N, int64_t n)
{
    int S = 1;
    while (S < 32 && wgrad_tiles(N) * S < 512 && tiles_of(n) / (2 * S) >= 2 * WWAVE) { S *= 2; }
    return S;
}

hipError_t launch_step_copies(const StepNet &N, hipStream_t s)
{
    hipLaunchKernelGGL(k_step_copies, dim3((unsigned)((N.npad + 255) / 256)), dim3(256), 0, s, N);
    return hipGetLastError();
}

hipError_t launch_step_grad(const StepNet &N, const StepBatch &B, const StepWork &w, hipStream_t s)
{
    const size_t lds = step_lds(N.d, N.H, N.Op);
    if (lds > STEP_LDS_MAX) { return hipErrorInvalidValue; }
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_step_tile), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { return e; }
    const int64_t tiles = tiles_of(B.n);
    hipLaunchKernelGGL(k_step_tile, dim3((unsigned)tiles), dim3(TPB), lds, s, N, B, w, 1.0f / (float)B.n);
    e = hipGetLastError();
    if (e != hipSuccess) { return e; }
    const WJob j1 = {w.X, w.dZ1, N.dp, N.Hp, N.d, N.H, N.oW1}, j2 = {w.H1, w.dZ2, N.Hp, N.Hp, N.H, N.H, N.oW2},
               j3 = {w.H2, w.dO, N.Hp, N.Op, N.H, N.Op, N.oW3};
    const int nb = (N.Op + 2 * N.Hp + 63) / 64;
    hipLaunchKernelGGL(k_step_wgrad, dim3((unsigned)(wgrad_tiles(N) + nb), (unsigned)step_splits(N, B.n)), dim3(WTPB), 0, s, j1, j2, j3, N,
                       w.bias, w.ws, tiles);
    return hipGetLastError();
}

hipError_t launch_step_sum(const StepNet &N, int64_t n, const StepWork &w, float *g, hipStream_t s)
{
    hipLaunchKernelGGL(k_step_adam<false>, dim3((unsigned)((N.npad + 255) / 256)), dim3(256), 0, s, N, w.ws, step_splits(N, n), g, nullptr,
                       nullptr, nullptr, nullptr, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f);
    return hipGetLastError();
}

hipError_t launch_step_adam(const StepNet &N, int64_t n, const StepWork &w, float *g, float *p, float *m, float *v, bf16_t *pb, float lr,
                            float b1, float b2, float eps, float bc1, float bc2, hipStream_t s)
{
    hipLaunchKernelGGL(k_step_adam<true>, dim3((unsigned)((N.npad + 255) / 256)), dim3(256), 0, s, N, w.ws, step_splits(N, n), g, p, m, v, pb,
                       lr, b1, b2, eps, bc1, bc2);
    return hipGetLastError();
}
} // namespace mcim
