// Sweep kernels for the RuNNer-style neural-network potential
// (src/EnergyEvaluation.jl:1182-1275, :1593-1621, :1735-1747, :1812-1822;
// MachineLearningPotential/{Cutoff,SymmFunc,DeltaMatrix}.jl).
//
// One workgroup owns one configuration for a whole cycle.  Its positions,
// feature matrix G (nf x atoms) and per-atom energies live in LDS.  A move
// builds the trial features D from G and the changes caused by moving atom i
// (radial terms by pair, angular terms by partner pair (j, k) with the
// exponentials shared by all functions of one eta), evaluates the network on D
// for every atom, and on acceptance swaps D and G.  Exchange, step adaptation and sampling run
// between cycles in nnp_cycle_kernel, so one launch of the sweep kernel is
// one cycle of every configuration.
#pragma once
#include "ptmc_surrogate.hpp"
#include "ptmc_sweep.hpp"

#include "ptmc_nnp_layout.hpp"

namespace ptmc {

struct NnpLds {
    float *X, *G, *D, *W1, *H1, *H2, *rn2, *fn, *ro2, *fo, *eat, *eatn;
    // tables copied from the host-prepared arrays: radial functions, angular
    // group descriptors and their waves, second-layer weights, b1 | b2 | w3
    float *rad, *W2, *B;
    int32_t *gd, *wg;
};

// static LDS holding the function tables (declared in each kernel)
#define NNP_TABLES_LDS                                                         \
    __shared__ float s_rad[4 * NNP_MAXF], s_w2[NNP_MAXH * NNP_MAXH], s_bias[3 * NNP_MAXH]; \
    __shared__ __align__(16) int32_t s_gdesc[NNP_MAXG * NNP_GD];              \
    __shared__ int32_t s_wgrp[(NNP_NT / 64) * (NNP_WG + 1)]

template <int NP>
__device__ inline NnpLds nnp_lds(float *base, int nf, int h1)
{
    NnpLds l;
    l.X = base;
    l.G = l.X + 3 * NP;
    l.D = l.G + nf * NP;
    l.W1 = l.D + nf * NP;
    l.H1 = l.W1 + nf * h1;
    l.H2 = l.H1 + NP * NNP_HS;
    l.rn2 = l.H2 + NP * NNP_HS;
    l.fn = l.rn2 + NP;
    l.ro2 = l.fn + NP;
    l.fo = l.ro2 + NP;
    l.eat = l.fo + NP;
    l.eatn = l.eat + NP;
    l.rad = l.W2 = l.B = nullptr;
    l.gd = l.wg = nullptr;
    return l;
}

// type-2 cutoff, MachineLearningPotential/Cutoff.jl:79-90
__device__ __forceinline__ float nnp_cutoff(float r, float rc) { return cutoff_cos2(r, rc); }

// (1 + lambda cos)^zeta of three cosines for zeta = 2^k: k squarings (k is
// uniform across the wave, so the loop is a scalar branch).
__device__ __forceinline__ void nnp_theta3(float lam, float kpow, float c0, float c1, float c2, float &p0,
                                           float &p1, float &p2)
{
    p0 = 1.0f + lam * c0;
    p1 = 1.0f + lam * c1;
    p2 = 1.0f + lam * c2;
    const int k = __builtin_amdgcn_readfirstlane((int)kpow);
    for (int s = 0; s < k; ++s) {
        p0 *= p0;
        p1 *= p1;
        p2 *= p2;
    }
}

// 1 / sqrt(x): the hardware's value (1 ulp) and one Newton step
__device__ __forceinline__ float nnp_rsq(float x)
{
    const float y = __builtin_amdgcn_rsqf(x);
    return y * __builtin_fmaf(-0.5f * x * y, y, 1.5f);
}

// number of set bits of a 64-lane mask below this lane
__device__ __forceinline__ int mbcnt64(uint64_t m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// cosines of the triangle (a, b, c) at a, b and c (Cutoff.jl:48-58)
__device__ __forceinline__ void nnp_angles(const float *a, const float *b, const float *c, float dab, float dac,
                                           float dbc, float &ta, float &tb, float &tc)
{
    const float abx = a[0] - b[0], aby = a[1] - b[1], abz = a[2] - b[2];
    const float acx = a[0] - c[0], acy = a[1] - c[1], acz = a[2] - c[2];
    const float bcx = b[0] - c[0], bcy = b[1] - c[1], bcz = b[2] - c[2];
    ta = (abx * acx + aby * acy + abz * acz) / (dab * dac);
    tb = (-abx * bcx - aby * bcy - abz * bcz) / (dab * dbc);
    tc = (acx * bcx + acy * bcy + acz * bcz) / (dac * dbc);
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// DPP lane permutation of a float (all 64 lanes active)
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Sum over each row of 16 lanes, left in every lane of the row: quad
// exchanges (quad_perm [1,0,3,2] and [2,3,0,1]), then half-row and row mirrors.
__device__ __forceinline__ float row_sum16(float v)
{
    v += dpp_f<0xB1>(v);
    v += dpp_f<0x4E>(v);
    v += dpp_f<0x141>(v);
    v += dpp_f<0x140>(v);
    return v;
}

// One eta group of angular functions as the move update reads it: e^{-eta x}
// = 2^{-eta2 x}; slots (lambda, k) = (+1, 0..4), (-1, 0..4); per slot tpz and
// the row (-1: none).
struct NnpGroup {
    float eta2;
    int row0;
    int top[2];  // per lambda: 1 + the highest power with a function (0: none)
    int rk[NNP_GMAX];
    float tpz[NNP_GMAX];
    __device__ void none()
    {
        eta2 = 0.0f;
        row0 = top[0] = top[1] = 0;
#pragma unroll
        for (int q = 0; q < NNP_GMAX; ++q) {
            rk[q] = -1;
            tpz[q] = 0.0f;
        }
    }
};

// Descriptor of group g from LDS in 16-byte reads; every word is uniform.
__device__ __forceinline__ void nnp_group(const int32_t *gd, int g, NnpGroup &G)
{
    int dw[NNP_GD];
#pragma unroll
    for (int u = 0; u < NNP_GD / 4; ++u) {
        const int4 w4 = reinterpret_cast<const int4 *>(gd + NNP_GD * g)[u];
        dw[4 * u] = w4.x;
        dw[4 * u + 1] = w4.y;
        dw[4 * u + 2] = w4.z;
        dw[4 * u + 3] = w4.w;
    }
    G.eta2 = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(dw[0]));
    G.row0 = __builtin_amdgcn_readfirstlane(dw[1]);
    G.top[0] = __builtin_amdgcn_readfirstlane(dw[2]) + 1;
    G.top[1] = __builtin_amdgcn_readfirstlane(dw[3]) + 1;
#pragma unroll
    for (int q = 0; q < NNP_GMAX; ++q) {
        G.tpz[q] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(dw[4 + q]));
        G.rk[q] = __builtin_amdgcn_readfirstlane(dw[4 + NNP_GMAX + q]);
    }
}

// Terms of one visit centred on one atom, both groups of the wave: e_new
// (1 + lambda c_new)^(2^k) + e_old (1 + lambda c_old)^(2^k) into slot (lambda,
// k) of a0 (a1), one squaring chain per lambda for both groups (eo carries the
// sign of the old term).  Every slot up to the highest power is added to: one
// without a function is never read, and a test per slot costs more than its
// two fma (a select each, its mask in a spilled scalar pair).
template <bool TWO>
__device__ __forceinline__ void nnp_terms(int top_p, int top_m, float cn, float co, float en0, float eo0, float en1,
                                          float eo1, float *a0, float *a1)
{
#pragma unroll
    for (int v = 0; v < 2; ++v) {
        const int top = v ? top_m : top_p;
        float pn = v ? 1.0f - cn : 1.0f + cn, po = v ? 1.0f - co : 1.0f + co;
#pragma unroll
        for (int k = 0; k < NNP_KSLOT; ++k) {
            if (k >= top) break;
            if (k > 0) {
                pn *= pn;
                po *= po;
            }
            const int q = v * NNP_KSLOT + k;
            a0[q] = __builtin_fmaf(en0, pn, a0[q]);
            a0[q] = __builtin_fmaf(eo0, po, a0[q]);
            if (TWO) {
                a1[q] = __builtin_fmaf(en1, pn, a1[q]);
                a1[q] = __builtin_fmaf(eo1, po, a1[q]);
            }
        }
    }
}

// m without its n lowest set bits (n up to their number): the position by
// halving over the bit counts
__device__ __forceinline__ uint64_t nnp_drop(uint64_t m, int n)
{
    int p = 0;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const int c = __popcll((m >> p) & ((1ull << s) - 1ull));
        const bool up = n >= c;
        n = up ? n - c : n;
        p = up ? p + s : p;
    }
    m = (m >> p) << p;
    return n > 0 ? m & (m - 1ull) : m;
}

// Adds one group's changes to the trial features D (which start as the
// current ones).  The 2^lp lanes of a target (an aligned block) combine their
// parts by quad exchanges and the half-row mirror, the first writes the
// target's entry.  The wave's sums of the terms centred on i go to the moved
// atom's column: the two row swaps merge the ten slots' registers into three
// (lambda by lane bit 5, the power's low bit by bit 4), so three row sums do
// for ten and one lane per slot writes.  Every old value is read before the
// first is written: the reads are in flight together.  All lanes call.
static_assert(NNP_KSLOT == 5, "slots (k, k + 1) of each lambda in three registers");
template <int NP, int SETS>
__device__ __forceinline__ void nnp_store(const NnpGroup &G, const int32_t *gd, int lp, bool writer, int j, int i,
                                          int lane, float *Dp, float *col, const float *aj, const float *ai)
{
    const float p1 = lp >= 1 ? 1.0f : 0.0f, p2 = lp >= 2 ? 1.0f : 0.0f, p3 = lp >= 3 ? 1.0f : 0.0f;
    // the slot whose sum this lane writes
    const int kq = 2 * (lane & 3) + ((lane >> 4) & 1), qi = NNP_KSLOT * (lane >> 5) + kq;
    const bool iw = (lane & 15) < 3 && kq < NNP_KSLOT;
    const int qc = iw ? qi : 0;
    const int irk = gd[4 + NNP_GMAX + qc];
    const float itpz = __int_as_float(gd[4 + qc]);
    float old[NNP_GMAX];
#pragma unroll
    for (int q = 0; q < NNP_GMAX; ++q) old[q] = Dp[(G.row0 + (G.rk[q] < 0 ? 0 : G.rk[q])) * NP + j];
    const int irow = G.row0 + (irk < 0 ? 0 : irk);
    float *di = Dp + irow * NP + i;
    const float oldi = SETS == 1 ? *di : 0.0f;
#pragma unroll
    for (int q = 0; q < NNP_GMAX; ++q) {
        if (G.rk[q] >= 0) {
            float v = aj[q];
            v = __builtin_fmaf(dpp_f<0xB1>(v), p1, v);
            v = __builtin_fmaf(dpp_f<0x4E>(v), p2, v);
            v = __builtin_fmaf(dpp_f<0x141>(v), p3, v);
            if (writer) Dp[(G.row0 + G.rk[q]) * NP + j] = __builtin_fmaf(v, G.tpz[q], old[q]);
        }
    }
    float h[NNP_KSLOT];
#pragma unroll
    for (int k = 0; k < NNP_KSLOT; ++k) h[k] = row_merge<32>(ai[k], ai[NNP_KSLOT + k]);
    const float s0 = row_sum16(row_merge<16>(h[0], h[1]));
    const float s1 = row_sum16(row_merge<16>(h[2], h[3]));
    const float s2 = row_sum16(row_pair_sum<16>(h[4]));
    const float s = (lane & 3) == 0 ? s0 : ((lane & 3) == 1 ? s1 : s2);
    if (iw && irk >= 0) {
        if (SETS == 1) *di = __builtin_fmaf(s, itpz, oldi);
        else col[irow] = s * itpz;  // the other half adds its own
    }
}

// Full feature matrix from positions into Gout (total_symm_calc,
// SymmFunc.jl:494-510; radial :259-278, angular :280-312).  All threads call.
template <int NP, int NT>
__device__ void nnp_full_build(const NnpTables &T, const NnpLds &L, float *Gout, int N)
{
    const int tid = threadIdx.x;
    for (int e = tid; e < T.nf * NP; e += NT) Gout[e] = 0.0f;
    __syncthreads();
    // radial: one (function, atom) per item
    for (int e = tid; e < T.n_rad_active * N; e += NT) {
        const int q = e / N, a = e % N;
        const float eta = L.rad[4 * q], norm = L.rad[4 * q + 1];
        const int row = (int)L.rad[4 * q + 2];
        float s = 0.0f;
        for (int b = 0; b < N; ++b) {
            if (b == a) continue;
            const float dx = L.X[a] - L.X[b], dy = L.X[NP + a] - L.X[NP + b], dz = L.X[2 * NP + a] - L.X[2 * NP + b];
            const float r2 = dx * dx + dy * dy + dz * dz;
            const float fc = nnp_cutoff(sqrtf(r2), T.r_cut);
            if (fc != 0.0f && fc != 1.0f) s += fc * expf(-eta * r2) * norm;
        }
        Gout[row * NP + a] = s;
    }
    // angular: one triangle a < b < c per item, all functions
    const int ntri = N * (N - 1) * (N - 2) / 6;
    for (int e = tid; e < ntri; e += NT) {
        // decode e -> (a, b, c)
        int a = 0, rem = e;
        while (rem >= (N - 1 - a) * (N - 2 - a) / 2) {
            rem -= (N - 1 - a) * (N - 2 - a) / 2;
            ++a;
        }
        int b = a + 1;
        while (rem >= N - 1 - b) {
            rem -= N - 1 - b;
            ++b;
        }
        const int c = b + 1 + rem;
        const float pa[3] = {L.X[a], L.X[NP + a], L.X[2 * NP + a]};
        const float pb[3] = {L.X[b], L.X[NP + b], L.X[2 * NP + b]};
        const float pc[3] = {L.X[c], L.X[NP + c], L.X[2 * NP + c]};
        auto d2 = [](const float *u, const float *v) {
            const float x = u[0] - v[0], y = u[1] - v[1], z = u[2] - v[2];
            return x * x + y * y + z * z;
        };
        const float rab = d2(pa, pb), rac = d2(pa, pc), rbc = d2(pb, pc);
        const float dab = sqrtf(rab), dac = sqrtf(rac), dbc = sqrtf(rbc);
        const float fp = nnp_cutoff(dab, T.r_cut) * nnp_cutoff(dac, T.r_cut) * nnp_cutoff(dbc, T.r_cut);
        if (fp == 0.0f) continue;
        float ta, tb, tc;
        nnp_angles(pa, pb, pc, dab, dac, dbc, ta, tb, tc);
        const float rs = rab + rac + rbc;
        for (int g = 0; g < T.n_groups; ++g) {
            const float ex = expf(-T.grp_eta[g] * rs) * fp;
            const int f0 = T.grp[2 * g], cnt = T.grp[2 * g + 1];
            for (int s = 0; s < cnt; ++s) {
                const int f = f0 + s;
                if (!T.abuild[f]) continue;
                const float lam = T.afn[4 * f], zc = T.afn[4 * f + 1], tpz = T.afn[4 * f + 2];
                const int row = (int)T.afn[4 * f + 3];
                float pa_, pb_, pc_;
                nnp_theta3(lam, zc, ta, tb, tc, pa_, pb_, pc_);
                atomicAdd(&Gout[row * NP + a], ex * pa_ * tpz);
                atomicAdd(&Gout[row * NP + b], ex * pb_ * tpz);
                atomicAdd(&Gout[row * NP + c], ex * pc_ * tpz);
            }
        }
    }
    __syncthreads();
    for (int e = tid; e < T.nf * N; e += NT) {
        const int q = e / N, a = e % N;
        Gout[q * NP + a] += T.row_off[q];
    }
    __syncthreads();
}

typedef float nnp_f32x4 __attribute__((ext_vector_type(4)));

// tanh x = 1 - 2 / (1 + e^{2x}), e^{2x} = 2^{2 log2(e) x} with the rounding
// of the argument put back (e^d = 1 + d) and the reciprocal refined by one
// Newton step: absolute error below 1.5e-7 over the whole range.  Past |x| =
// 40 the value is +-1 in binary32 at any rate; the clamp keeps e finite there.
__device__ __forceinline__ float nnp_tanh(float x)
{
    const float c = 2.8853900817779268f, x1 = x > 40.0f ? 40.0f : (x < -40.0f ? -40.0f : x);
    const float t = x1 * c, d = __builtin_fmaf(x1, c, -t) * 0.6931471805599453f;
    float e = __builtin_amdgcn_exp2f(t);
    e = __builtin_fmaf(e, d, e) + 1.0f;
    const float y = __builtin_amdgcn_rcpf(e);
    return __builtin_fmaf(-2.0f, __builtin_fmaf(__builtin_fmaf(-e, y, 1.0f), y, y), 1.0f);
}

// One 16 x 16 tile (atoms r0 .., outputs c0 ..) of a layer's product over n
// inputs, binary32 on the matrix cores: lane l feeds A[row l % 16][k l / 16]
// from x(k, row) and B[k l / 16][column l % 16] from w(k, column); value v of
// the result belongs to row 4 (l / 16) + v, column l % 16.  Four partial sums:
// independent steps, and a quarter of the terms in each rounding chain.
template <typename X, typename W>
__device__ __forceinline__ nnp_f32x4 nnp_tile(int n, X x, W w)
{
    const int lk = (threadIdx.x & 63) >> 4;
    nnp_f32x4 z[4] = {};
    int k0 = 0;
    auto block = [&](auto steps) {  // the operands of all steps in flight together
        constexpr int S = decltype(steps)::value;
        float a[S], b[S];
#pragma unroll
        for (int u = 0; u < S; ++u) {
            a[u] = x(k0 + 4 * u + lk);
            b[u] = w(k0 + 4 * u + lk);
        }
#pragma unroll
        for (int u = 0; u < S; ++u) z[u & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], z[u & 3], 0, 0, 0);
        k0 += 4 * S;
    };
    while (k0 + 32 <= n) block(std::integral_constant<int, 8>{});
    if (k0 + 16 <= n) block(std::integral_constant<int, 4>{});
    if (k0 + 8 <= n) block(std::integral_constant<int, 2>{});
    for (; k0 < n; k0 += 4) {
        const int k = k0 + lk, kc = k < n ? k : n - 1;
        const float m = k < n ? 1.0f : 0.0f;
        z[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x(kc) * m, w(kc) * m, z[3], 0, 0, 0);
    }
    return (z[0] + z[1]) + (z[2] + z[3]);
}

// Per-atom network energies of the features Gin into out[N]
// (n_features -> tanh h1 -> tanh h2 -> linear 1, ForwardPass.jl:23-39).
// The two hidden layers are products on the matrix cores in binary32, a 16 x 16
// tile per wave (64 atoms x 32 outputs are eight tiles; two waves with 32 x 32
// tiles left the other six waiting for 44 steps of 64 cycles).  The
// output layer's dot product is a row sum per tile; the FP64 total is a sum
// over each wave of 64 atoms (DPP and row swaps), then the waves' sums in order.  All threads call.
template <int NP, int NT>
__device__ void nnp_forward(const NnpTables &T, const NnpLds &L, const float *Gin, int N, float *out,
                            double *total = nullptr)
{
    constexpr int NW = NP / 64;
    __shared__ double s_fpart[NNP_NP_WIDE / 64];
    const int tid = threadIdx.x, l = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = l & 15, lk = l >> 4;
    const int nf = T.nf, h1 = T.h1, h2 = T.h2;
    for (int t = w; t < 2 * (NP / 16); t += NT / 64) {
        const int r0 = 16 * (t % (NP / 16)), c0 = 16 * (t / (NP / 16));
        if (r0 >= N || c0 >= h1) continue;
        const int c = c0 + lr, cc = c < h1 ? c : h1 - 1;
        const nnp_f32x4 z = nnp_tile(nf, [&](int k) { return Gin[k * NP + r0 + lr]; },
                                     [&](int k) { return L.W1[k * h1 + cc]; });
        if (c < h1) {
            const float bias = L.B[c];
#pragma unroll
            for (int v = 0; v < 4; ++v) L.H1[(r0 + 4 * lk + v) * NNP_HS + c] = nnp_tanh(z[v] + bias);
        }
    }
    __syncthreads();
    for (int t = w; t < 2 * (NP / 16); t += NT / 64) {
        const int r0 = 16 * (t % (NP / 16)), c0 = 16 * (t / (NP / 16));
        if (r0 >= N || c0 >= h2) continue;
        const int c = c0 + lr, cc = c < h2 ? c : h2 - 1;
        const nnp_f32x4 z = nnp_tile(h1, [&](int k) { return L.H1[(r0 + lr) * NNP_HS + k]; },
                                     [&](int k) { return L.W2[k * h2 + cc]; });
        float bias = 0.0f, w3 = 0.0f;
        if (c < h2) {
            bias = L.B[NNP_MAXH + c];
            w3 = L.B[2 * NNP_MAXH + c];
        }
        // second hidden layer times the output weights, summed over the tile's
        // columns (w3 = 0 past the last)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float y = row_sum16(nnp_tanh(z[v] + bias) * w3);
            if (lr == 0) L.H2[(c0 >> 4) * NP + r0 + 4 * lk + v] = y;
        }
    }
    __syncthreads();
    if (w < NW) {
        const int at = 64 * w + l;
        float y = 0.0f;
        if (at < N) {
            y = L.H2[at];
            if (h2 > 16) y += L.H2[NP + at];
            y += T.b3;
            out[at] = y;
        }
        // FP64 total of the atomic energies
        if (total != nullptr) {
            double t = at < N ? (double)y : 0.0;
            t = group_sum<16>(t);
            t += row_xor<16>(t);
            t += row_xor<32>(t);
            if (NW == 1 && l == 0) *total = t;
            if (NW > 1 && l == 0) s_fpart[w] = t;
        }
    }
    if (NW > 1 && total != nullptr) {
        __syncthreads();
        if (tid == 0) {
            double t = s_fpart[0];
            for (int v = 1; v < NW; ++v) t += s_fpart[v];
            *total = t;
        }
    }
    __syncthreads();
}

template <int NP, int NT>
__device__ __forceinline__ void nnp_load(const SweepArgs &a, const NnpLds &L, int slot)
{
    const NnpTables &T = a.nnp;
    const float *gX = reinterpret_cast<const float *>(a.coords) + (size_t)slot * 3 * NP;
    const int tid = threadIdx.x;
    for (int e = tid; e < 3 * NP; e += NT) L.X[e] = gX[e];
    for (int e = tid; e < T.nf * T.h1; e += NT) L.W1[e] = T.w1[e];
    for (int e = tid; e < 4 * T.n_rad_active; e += NT) L.rad[e] = T.rad[e];
    for (int e = tid; e < NNP_GD * T.n_groups; e += NT) L.gd[e] = T.gdesc[e];
    for (int e = tid; e < (NNP_NT / 64) * (NNP_WG + 1); e += NT) L.wg[e] = T.wgroups[e];
    for (int e = tid; e < T.h1 * T.h2; e += NT) L.W2[e] = T.w2[e];
    for (int e = tid; e < NNP_MAXH; e += NT) {
        L.B[e] = e < T.h1 ? T.b1[e] : 0.0f;
        L.B[NNP_MAXH + e] = e < T.h2 ? T.b2[e] : 0.0f;
        L.B[2 * NNP_MAXH + e] = e < T.h2 ? T.w3[e] : 0.0f;
    }
}

#define NNP_BIND_TABLES(L) \
    L.rad = s_rad;         \
    L.W2 = s_w2;           \
    L.B = s_bias;          \
    L.gd = s_gdesc;        \
    L.wg = s_wgrp

// set_variables + initialise_energy (src/EnergyEvaluation.jl:1812-1822,
// :1735-1747): features, per-atom energies and the FP64 total of each slot.
template <int NP, int NT>
__global__ void __launch_bounds__(NT) nnp_init_kernel(SweepArgs a)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const NnpTables &T = a.nnp;
    const int slot = blockIdx.x;
    if (a.init_run >= 0 && a.slot_run[slot] != a.init_run) return;  // whole workgroup
    NNP_TABLES_LDS;
    NnpLds L = nnp_lds<NP>(reinterpret_cast<float *>(lds_raw), T.nf, T.h1);
    NNP_BIND_TABLES(L);
    const int N = a.runs[a.slot_run[slot]].n_atoms;
    nnp_load<NP, NT>(a, L, slot);
    __syncthreads();
    nnp_full_build<NP, NT>(T, L, L.G, N);
    __shared__ double s_tot;
    nnp_forward<NP, NT>(T, L, L.G, N, L.eat, &s_tot);
    float *gG = a.feat + (size_t)slot * T.nf * NP;
    for (int e = threadIdx.x; e < T.nf * NP; e += NT) gG[e] = L.G[e];
    for (int e = threadIdx.x; e < NP; e += NT) a.eatom[(size_t)slot * NP + e] = e < N ? L.eat[e] : 0.0f;
    if (threadIdx.x == 0) a.slot_en[slot] = s_tot;
}

// One Monte-Carlo cycle (N moves) of one configuration per workgroup
// (mc_step!, src/MCRun.jl:169-182, with energy_update!(RuNNerPotential)).
// DA: delayed acceptance with the learned surrogate (one workgroup per CU by
// LDS, so the register budget is relaxed for that variant).  NP: atoms of a
// slot, 64 or 128 (the near atoms of a move are then up to 127, their partner
// masks two words).  NT: 512 threads, or 1024 where a workgroup has a CU to
// itself (always with NP = 128): the second half's waves own the same groups as
// the first's and take every other target, their sums at the moved atom are
// added after the visits.
//
// Bound by instruction issue in the angular visits (a 55-atom move visits about
// 1000 triangles from two of their atoms, once per group pair): 28,000 of a
// move's 51,000 cycles with one workgroup of 512 threads on a CU.  A visit's
// instructions went from about 330 to 190: the lane's share of the partners is
// cut from the mask once per target (not popped past on every visit), cosines
// from unit vectors in place of IEEE divides and roots, one squaring chain for
// both groups of a wave, no select per slot.  Store: sums merged across rows
// before they are summed, 20 wave sums as 6 row sums, and the lanes of a target
// added by one fma each.  us per cycle of 40 temperatures x 55 atoms (8 + 80
// functions) 2070 before, 1210 so, 1117 on 1024 threads; of 1280 configurations
// 6900, 3950, 3740 with the visits split by their terms; of 20 x 78 atoms 3000,
// 1970, 1665 on 1024 threads.
template <bool DA, int NP, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(DA ? 2 : 4)))
nnp_sweep_kernel(SweepArgs a)
{
    static_assert(NT == NNP_NT || (NT == 2 * NNP_NT && !DA), "one or two workgroup halves");
    static_assert(NP == NNP_NP || (NP == NNP_NP_WIDE && NT == 2 * NNP_NT), "the targets of a half fit a wave");
    constexpr int SETS = NT / NNP_NT;  // halves of the workgroup, each with every other near atom as its targets
    constexpr int NW = NP / 64;  // 64-bit words of an atom mask
    constexpr bool SPLIT = NW == 1;  // visits with and without the terms at i apart
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ int s_flag, s_err, s_nnear;
    __shared__ uint64_t s_wmask[NW];
    __shared__ uint8_t s_near[NP];
    __shared__ double s_en;
    __shared__ float s_trial[3], s_old[3];
    const NnpTables &T = a.nnp;
    const int slot = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    NNP_TABLES_LDS;
    NnpLds L = nnp_lds<NP>(reinterpret_cast<float *>(lds_raw), T.nf, T.h1);
    NNP_BIND_TABLES(L);
    const RunInfo &ri = a.runs[a.slot_run[slot]];
    const int N = ri.n_atoms;
    const uint32_t nsteps = (uint32_t)N;
    const int t = a.slot_temp[slot];
    const int Tg = ri.temp_base + t;
    const uint32_t sweep = (uint32_t)a.sweep0;
    const double beta = a.t_beta[Tg];
    const float delta_r = (float)a.t_displ[2 * Tg];
    const float radius2 = (float)ri.radius2;

    nnp_load<NP, NT>(a, L, slot);
    const float *gG = a.feat + (size_t)slot * T.nf * NP;
    for (int e = tid; e < T.nf * NP; e += NT) L.G[e] = gG[e];
    for (int e = tid; e < NP; e += NT) L.eat[e] = a.eatom[(size_t)slot * NP + e];
    double E = a.slot_en[slot];
    if (tid == 0) s_err = 0;
    // delayed acceptance: surrogate descriptors and atom energies in LDS
    // (rebuilt from the positions at every launch)
    __shared__ float s_acci[SUR_K];
    __shared__ double s_ehat;
    constexpr bool da = DA;
    float *Sd = nullptr, *Sn = nullptr, *sat = nullptr, *satn = nullptr, *sgeo = nullptr;
    SurNet net{};
    const SurGeom sg = sur_geom(a.sur_rcut);
    double Ehat = 0.0;
    long long n_prop = 0, n_acc1 = 0;
    if (da) {
        float *base = reinterpret_cast<float *>(lds_raw) + nnp_lds_floats(T.nf, T.h1);
        Sd = base;
        Sn = Sd + NP * SUR_SS;
        net.W1 = reinterpret_cast<short *>(Sn + NP * SUR_SS);
        net.W2 = net.W1 + SUR_K * SUR_H;
        net.Hb = net.W2 + SUR_H * SUR_H;
        sat = reinterpret_cast<float *>(net.Hb + NP * SUR_HS);
        satn = sat + NP;
        net.b1 = satn + NP;
        net.b2 = net.b1 + SUR_H;
        net.w3 = net.b2 + SUR_H;
        sgeo = net.w3 + SUR_H;  // per atom: r_new, r_old, f_c(r_new), f_c(r_old)
        sur_load_net(net, a.sur_w, NT);
        sur_descriptors(sg, L.X, N, Sd, SUR_SS, NT);
        for (int e = tid; e < NP * SUR_SS; e += NT) Sn[e] = 0.0f;
        __syncthreads();
        sur_atom_energies(net, Sd, N, L.H1, sat, &s_ehat);
        Ehat = s_ehat;
    }
    __syncthreads();
    int nacc = 0;
    // current features and the scratch that becomes the trial features; an
    // accepted move swaps the two (swap_vars!(NNPVariables), src/swap_config.jl:213-221)
    float *Gp = L.G, *Dp = L.D;
    // scratch in H1 until the network pass: partner masks [near atom][NW words],
    // lane tables of the waves, and with two halves their sums at the moved atom
    uint64_t *s_mask = reinterpret_cast<uint64_t *>(L.H1);
    uint16_t *s_lt = reinterpret_cast<uint16_t *>(L.H1 + 2 * NW * NP) + 64 * (tid >> 6);
    float *s_col = L.H1 + 2 * NW * NP + 32 * (NT / 64);
    static_assert(2 * NW * NP + 32 * (NT / 64) + (SETS > 1 ? SETS * NNP_MAXF : 0) <= NP * NNP_HS, "H1 holds the scratch");
    // 16-byte aligned by its offset, so that the compiler still sees an LDS
    // address (a pointer through an integer is read with flat loads)
    float *nb_base = reinterpret_cast<float *>(lds_raw) + (((int)(L.H2 - reinterpret_cast<float *>(lds_raw)) + 3) & ~3);
    float4 *nb_a = reinterpret_cast<float4 *>(nb_base);
    float4 *nb_b = nb_a + NP, *nb_u = nb_b + NP, *nb_v = nb_u + NP;
    // near atom q of the list (atom j): {x, y, z, f_new}, {r2_new, r2_old,
    // f_old, -} and the unit vectors from the moved atom's new and old position
    auto pack = [&](int q, int j, const float (&pt)[3], const float (&po)[3]) {
        const float x = L.X[j], y = L.X[NP + j], z = L.X[2 * NP + j], rn = L.rn2[j], ro = L.ro2[j];
        const float un = nnp_rsq(rn), uo = nnp_rsq(ro);
        nb_a[q] = make_float4(x, y, z, L.fn[j]);
        nb_b[q] = make_float4(rn, ro, L.fo[j], 0.0f);
        nb_u[q] = make_float4((x - pt[0]) * un, (y - pt[1]) * un, (z - pt[2]) * un, 0.0f);
        nb_v[q] = make_float4((x - po[0]) * uo, (y - po[1]) * uo, (z - po[2]) * uo, 0.0f);
    };

    for (uint32_t m = 0; m < nsteps; ++m) {
        // draws and trial position (every thread the same), src/MCMoves.jl:115-135
        MoveDraw<float> d0 = move_draw<float>(a.seed, ri.run_key, (uint32_t)t, sweep, m, 0u, nsteps);
        const int i = (int)d0.index;
        float xi = L.X[i], yi = L.X[NP + i], zi = L.X[2 * NP + i];
        float tx, ty, tz;
        make_trial<float, BC_SPHERE, false>(xi, yi, zi, d0, delta_r, 0.0f, 0.0f, tx, ty, tz);
        if (outside_sphere<float>(tx, ty, tz, radius2)) {
            int count = 0;
            uint32_t attempt = 0;
            while (outside_sphere<float>(tx, ty, tz, radius2)) {
                count += 1;
                if (count == 50) {
                    __syncthreads();
                    if (tid == 0) {
                        double c[3] = {0.0, 0.0, 0.0};
                        for (int b = 0; b < N; ++b)
                            for (int k = 0; k < 3; ++k) c[k] += (double)L.X[k * NP + b];
                        for (int k = 0; k < 3; ++k) c[k] /= (double)N;
                        for (int b = 0; b < N; ++b)
                            for (int k = 0; k < 3; ++k)
                                L.X[k * NP + b] = (float)((double)L.X[k * NP + b] - c[k]);
                    }
                    __syncthreads();
                } else {
                    attempt += 1;
                    MoveDraw<float> dd = move_draw<float>(a.seed, ri.run_key, (uint32_t)t, sweep, m, attempt, nsteps);
                    xi = L.X[i];
                    yi = L.X[NP + i];
                    zi = L.X[2 * NP + i];
                    make_trial<float, BC_SPHERE, false>(xi, yi, zi, dd, delta_r, 0.0f, 0.0f, tx, ty, tz);
                    if (count == 100) {
                        if (tid == 0) s_err = 1;
                        break;
                    }
                }
            }
            xi = L.X[i];
            yi = L.X[NP + i];
            zi = L.X[2 * NP + i];
        }
        const float pt[3] = {tx, ty, tz}, po[3] = {xi, yi, zi};
        // distances and cutoffs to the new and old position; hard-core test
        // (one lane per atom) and the list of the atoms within the cut-off of
        // either position, the only partners of angular terms, in atom order
        if (tid == 0) s_flag = 0;
        __syncthreads();
        if (tid < NP) {
            const int j = tid;
            bool near = false;
            if (j < N) {
                const float px = L.X[j], py = L.X[NP + j], pz = L.X[2 * NP + j];
                float dx = tx - px, dy = ty - py, dz = tz - pz;
                const float rn = j == i ? 0.0f : dx * dx + dy * dy + dz * dz;
                dx = xi - px;
                dy = yi - py;
                dz = zi - pz;
                const float ro = j == i ? 0.0f : dx * dx + dy * dy + dz * dz;
                const float fnj = nnp_cutoff(sqrtf(rn), T.r_cut), foj = nnp_cutoff(sqrtf(ro), T.r_cut);
                L.rn2[j] = rn;
                L.ro2[j] = ro;
                L.fn[j] = fnj;
                L.fo[j] = foj;
                if (j != i && (double)rn < T.hardcore2) s_flag = 1;
                near = j != i && (fnj != 0.0f || foj != 0.0f);
            }
            const uint64_t b = __ballot(near);
            if constexpr (NW == 1) {
                if (near) {
                    // packed per near atom for the angular visits (in the H2 scratch)
                    const int q = mbcnt64(b);
                    s_near[q] = (uint8_t)j;
                    pack(q, j, pt, po);
                }
                if (lane == 0) s_nnear = __popcll(b);
            } else {
                if (lane == 0) s_wmask[tid >> 6] = b;
            }
        }
        if constexpr (NW > 1) {
            // the near atoms of lower waves come first: list positions from
            // the waves' masks once every wave has written its own
            __syncthreads();
            if (tid < NP) {
                const int j = tid;
                const uint64_t b = s_wmask[tid >> 6];
                if ((b >> lane) & 1ull) {
                    int q = mbcnt64(b);
                    for (int v = 0; v < (tid >> 6); ++v) q += __popcll(s_wmask[v]);
                    s_near[q] = (uint8_t)j;
                    pack(q, j, pt, po);
                }
            }
            if (tid == 0) {
                int t = 0;
                for (int v = 0; v < NW; ++v) t += __popcll(s_wmask[v]);
                s_nnear = t;
            }
        }
        // trial features start as the current ones; every changed entry is
        // written once, as current plus change
        for (int e = tid; e < T.nf * NP / 4; e += NT)
            reinterpret_cast<float4 *>(Dp)[e] = reinterpret_cast<const float4 *>(Gp)[e];
        if (SETS > 1 && tid < SETS * NNP_MAXF) s_col[tid] = 0.0f;
        if (da && tid < SUR_K) s_acci[tid] = 0.0f;
        __syncthreads();
        // delayed acceptance, stage 1: Metropolis on the surrogate energy change
        bool stage1 = true;
        double dEh = 0.0, Ehn = 0.0;
        if (da) {
            // distances and cutoffs of every atom to the two positions, once
            if (tid < N) {
                const float rn = sqrtf(L.rn2[tid]), ro = sqrtf(L.ro2[tid]);
                sgeo[tid] = rn;
                sgeo[NP + tid] = ro;
                sgeo[2 * NP + tid] = tid == i ? 0.0f : sur_cutoff(rn, sg.r_cut);
                sgeo[3 * NP + tid] = tid == i ? 0.0f : sur_cutoff(ro, sg.r_cut);
            }
            __syncthreads();
            float accq = 0.0f;
            const int kq = tid & (SUR_K - 1);  // NT is a multiple of SUR_K: fixed k per thread
            const float mu = sur_mu(sg, kq);
            for (int j = tid / SUR_K; j < N; j += NT / SUR_K) {
                if (j == i) continue;
                const float fcn = sgeo[2 * NP + j], fco = sgeo[3 * NP + j];
                const float pn = sur_phi_mu(sg, sgeo[j], fcn, mu);
                const float pq = sur_phi_mu(sg, sgeo[NP + j], fco, mu);
                Sn[j * SUR_SS + kq] = __builtin_fmaf(SUR_SIN, pn - pq, Sd[j * SUR_SS + kq]);
                accq += pn;
            }
            atomicAdd(&s_acci[kq], accq);
            __syncthreads();
            if (tid < SUR_K) Sn[i * SUR_SS + tid] = SUR_SIN * s_acci[tid];
            __syncthreads();
            sur_atom_energies(net, Sn, N, L.H1, satn, &s_ehat);
            Ehn = s_ehat;
            dEh = Ehn - Ehat;
            stage1 = (dEh <= 0.0) || (det_exp(-dEh * beta) >= (double)d0.umet);
            n_prop += 1;
            n_acc1 += stage1 ? 1 : 0;
        }
        double new_en = 100.0;  // the hard-core sentinel, src/EnergyEvaluation.jl:1604-1606
        if (da && !stage1) new_en = __builtin_nan("");
        if (stage1 && !s_flag) {
            if constexpr (DA) {
                // the surrogate's layer scratch covered the packed near-atom data
                if (tid < s_nnear) pack(tid, s_near[tid], pt, po);
                __syncthreads();
            }
            // radial changes, DeltaMatrix.jl:794-822: one wave per function,
            // one lane per atom (NW atoms per lane in the wide layout)
            for (int q = tid >> 6; q < T.n_rad_active; q += NT / 64) {
                const float eta = L.rad[4 * q], norm = L.rad[4 * q + 1];
                const int row = (int)L.rad[4 * q + 2];
                float dsum = 0.0f;
#pragma unroll
                for (int v = 0; v < NW; ++v) {
                    const int at = 64 * v + lane;
                    float d = 0.0f;
                    if (at < N && at != i)
                        d = expf(-eta * L.rn2[at]) * (L.fn[at] * norm) + expf(-eta * L.ro2[at]) * (-L.fo[at] * norm);
                    if (at < N && at != i) Dp[row * NP + at] = Gp[row * NP + at] + d;
                    dsum += d;
                }
                const float s = wave_sum(dsum);
                if (lane == 0) Dp[row * NP + i] = Gp[row * NP + i] + s;
            }
            // angular changes, DeltaMatrix.jl:827-872.  Every partner pair
            // (j, k) of the moved atom i whose triangle lies inside the cut-off
            // (old or new position) is visited from j and from k; a visit adds
            // the terms centred on its own atom and, from the atom of smaller
            // index, the terms centred on i.  Each wave owns a few eta groups
            // (their feature rows), each lane one target atom j (or a half or
            // quarter of its partners when few atoms are near), so every
            // feature entry is written by one lane with a plain store: no LDS
            // atomics (float LDS adds run far below the store rate).
            const int n_near = s_nnear;
            const float rc2 = T.r_cut * T.r_cut * 1.0001f;  // loose: the cut-off function decides below
            for (int a = tid >> 6; a < n_near; a += NT / 64) {
                const float4 pa = nb_a[a];
                const float foa = nb_b[a].z;
#pragma unroll
                for (int v = 0; v < NW; ++v) {
                    const int b = 64 * v + lane;
                    bool act = false;
                    if (b < n_near && b != a) {
                        const float4 pb = nb_a[b];
                        if (pa.w * pb.w != 0.0f || foa * nb_b[b].z != 0.0f) {
                            const float dx = pa.x - pb.x, dy = pa.y - pb.y, dz = pa.z - pb.z;
                            act = dx * dx + dy * dy + dz * dz < rc2;
                        }
                    }
                    const uint64_t m = __ballot(act);
                    if (lane == 0) s_mask[a * NW + v] = m;
                }
            }
            __syncthreads();
            // Lanes per target: target a gets P_a = 1, 2, 4 or 8 lanes, the fewest
            // that bring its share of visits down to the load T, T the smallest
            // load for which the shares fit 64 lanes (bisection, the lane count
            // summed by ballots).  Blocks of P lanes are laid out by P (8, 4, 2,
            // 1), so each is aligned for the quad and half-row exchanges that
            // combine them.  Every wave builds the same tables (of its half's
            // targets) in its own LDS slice: no barrier needed within a wave.
            // uniform over the wave, and said so: the loops over groups and
            // powers then branch on scalars
            const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int set = w / (NNP_NT / 64), wl = w % (NNP_NT / 64);
            const int nc = (n_near - set + SETS - 1) / SETS;  // entry e: near atom SETS e + set
            int used = 0;
            {
                int La = 0;
                if (lane < nc) {
#pragma unroll
                    for (int v = 0; v < NW; ++v) La += __popcll(s_mask[(SETS * lane + set) * NW + v]);
                }
                // lanes of a target at load T: 1 up to T visits, 2 up to 2 T,
                // 4 up to 4 T, else 8; their sum over the targets
                auto lanes_used = [&](int load) {
                    return nc + __popcll(__ballot(La > load)) + 2 * __popcll(__ballot(La > 2 * load)) +
                           4 * __popcll(__ballot(La > 4 * load));
                };
                int lo = 1, hi = 64 * NW;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (lanes_used(mid) <= 64) hi = mid;
                    else lo = mid + 1;
                }
                const int Pa = lane >= nc ? 0 : (La <= lo ? 1 : (La <= 2 * lo ? 2 : (La <= 4 * lo ? 4 : 8)));
#pragma unroll
                for (int cc = 3; cc >= 0; --cc) {
                    const bool in = Pa == (1 << cc);
                    const uint64_t b = __ballot(in);
                    if (in)
                        for (int q = 0; q < Pa; ++q)
                            s_lt[used + (mbcnt64(b) << cc) + q] = (uint16_t)(lane | (q << 6) | (cc << 9));
                    used += __popcll(b) << cc;
                }
            }
            // this lane's target: lanes, part, atom, the partners of its part with
            // which the visit also carries the terms centred on i (o) and the
            // others (m), packed data.  Of the n near atoms in a circle, a target
            // carries those terms for the (n - 1) / 2 after it (and of an opposite
            // pair the first does): every target for about half of its partners,
            // so the lanes of a wave do such visits together, and then the
            // others.  Slots of 128 atoms go through all partners at once and
            // test each (o holds the circle): with two mask words and 26 functions
            // the cut costs more than it saves (20 x 78 atoms 1.83 ms split, 1.66
            // so; 1280 x 55 atoms, 88 functions, 3.95 unsplit, 3.72 split).
            struct Target {
                int lp, part, j;
                bool tact;
                uint64_t m0, m1, o0, o1;
                float4 ja, jb, ju, jv;
            };
            auto target = [&]() {
                Target g;
                const int ent = lane < used ? (int)s_lt[lane] : 0;
                g.lp = ent >> 9;
                const int ta = SETS * (ent & 63) + set;
                g.part = (ent >> 6) & 7;
                g.tact = lane < used;
                g.j = g.tact ? (int)s_near[ta] : 0;
                uint64_t m0 = g.tact ? s_mask[ta * NW] : 0ull, m1 = 0ull;
                if constexpr (NW > 1) m1 = g.tact ? s_mask[ta * NW + 1] : 0ull;
                // list indices ta + 1 .. ta + h round the circle of n_near
                const int h = (n_near - 1) / 2 + (((n_near & 1) == 0 && 2 * ta < n_near) ? 1 : 0);
                const int end = ta + 1 + h;  // past n_near: the rest from 0
                auto below = [](int b, int word) {  // bits of a word whose index is below b
                    const int k = b - 64 * word;
                    return k <= 0 ? 0ull : (k >= 64 ? ~0ull : (1ull << k) - 1ull);
                };
                auto circle = [&](int word) {
                    const uint64_t up = below(end, word) & ~below(ta + 1, word);
                    return end > n_near ? up | below(end - n_near, word) : up;
                };
                const uint64_t c0 = circle(0), c1 = NW > 1 ? circle(1) : 0ull;
                g.o0 = SPLIT ? m0 & c0 : c0;
                g.o1 = SPLIT ? m1 & c1 : c1;
                g.m0 = SPLIT ? m0 & ~c0 : m0;
                g.m1 = SPLIT ? m1 & ~c1 : m1;
                // the part's share: equal counts, by rank among the partners
                auto share = [&](uint64_t &a0, uint64_t &a1, int part) {
                    const int n0 = __popcll(a0), n = n0 + (NW > 1 ? __popcll(a1) : 0);
                    const int r0 = (part * n) >> g.lp, r1 = ((part + 1) * n) >> g.lp;
                    auto cut_word = [](uint64_t m, int c, int a, int b) {  // bits of rank a .. b - 1 of c
                        a = a < 0 ? 0 : (a < c ? a : c);
                        b = b < 0 ? 0 : (b < c ? b : c);
                        return nnp_drop(m, a) & ~nnp_drop(m, b);
                    };
                    if constexpr (NW > 1) a1 = cut_word(a1, n - n0, r0 - n0, r1 - n0);
                    a0 = cut_word(a0, n0, r0, r1);
                };
                if constexpr (SPLIT) share(g.o0, g.o1, g.part);
                share(g.m0, g.m1, g.part);
                g.ja = nb_a[ta];
                g.jb = nb_b[ta];
                g.ju = nb_u[ta];
                g.jv = nb_v[ta];
                return g;
            };
            const Target tg = target();  // read once for all group passes
            const int ngw = __builtin_amdgcn_readfirstlane(L.wg[wl * (NNP_WG + 1)]);
            for (int gi = 0; gi < ngw; gi += 2) {
                // up to two groups per pass over the visits
                const int ga = __builtin_amdgcn_readfirstlane(L.wg[wl * (NNP_WG + 1) + 1 + gi]);
                const int gb = gi + 1 < ngw ? __builtin_amdgcn_readfirstlane(L.wg[wl * (NNP_WG + 1) + 2 + gi]) : -1;
                NnpGroup G0, G1;
                nnp_group(L.gd, ga, G0);
                if (gb >= 0) nnp_group(L.gd, gb, G1);
                else G1.none();
                const int top_p = G0.top[0] > G1.top[0] ? G0.top[0] : G1.top[0];
                const int top_m = G0.top[1] > G1.top[1] ? G0.top[1] : G1.top[1];
                {
                    const float4 ja = tg.ja, jb = tg.jb, ju = tg.ju, jv = tg.jv;
                    float aj0[NNP_GMAX], ai0[NNP_GMAX], aj1[NNP_GMAX], ai1[NNP_GMAX];
#pragma unroll
                    for (int q = 0; q < NNP_GMAX; ++q) aj0[q] = ai0[q] = aj1[q] = ai1[q] = 0.0f;
                    auto visits = [&](auto two, auto own, uint64_t m0, uint64_t m1) {
                        constexpr bool TWO = decltype(two)::value;
                        while (NW == 1 ? m0 != 0ull : (m0 | m1) != 0ull) {
                            int bk;
                            bool at_i = decltype(own)::value;
                            if (NW == 1 || m0 != 0ull) {
                                bk = __builtin_ctzll(m0);
                                m0 &= m0 - 1ull;
                                if (!SPLIT) at_i = ((tg.o0 >> bk) & 1ull) != 0ull;
                            } else {
                                bk = __builtin_ctzll(m1);
                                m1 &= m1 - 1ull;
                                if (!SPLIT) at_i = ((tg.o1 >> bk) & 1ull) != 0ull;
                                bk += 64;
                            }
                            const float4 ka = nb_a[bk], kb = nb_b[bk];
                            const float dx = ja.x - ka.x, dy = ja.y - ka.y, dz = ja.z - ka.z;
                            const float rjk = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                            const float ijk = nnp_rsq(rjk);
                            const float fjk = nnp_cutoff(rjk * ijk, T.r_cut);
                            const float fpn = ja.w * ka.w * fjk, fpo = jb.z * kb.z * fjk;
                            if (fpn == 0.0f && fpo == 0.0f) continue;
                            const float rsn = jb.x + kb.x + rjk, rso = jb.y + kb.y + rjk;
                            // cosines at j, new and old, from the unit vectors i -> j and k -> j
                            const float cjn = __builtin_fmaf(ju.z, dz, __builtin_fmaf(ju.y, dy, ju.x * dx)) * ijk;
                            const float cjo = __builtin_fmaf(jv.z, dz, __builtin_fmaf(jv.y, dy, jv.x * dx)) * ijk;
                            const float en0 = __builtin_amdgcn_exp2f(-G0.eta2 * rsn) * fpn;
                            const float eo0 = -(__builtin_amdgcn_exp2f(-G0.eta2 * rso) * fpo);
                            float en1 = 0.0f, eo1 = 0.0f;
                            if (TWO) {
                                en1 = __builtin_amdgcn_exp2f(-G1.eta2 * rsn) * fpn;
                                eo1 = -(__builtin_amdgcn_exp2f(-G1.eta2 * rso) * fpo);
                            }
                            nnp_terms<TWO>(top_p, top_m, cjn, cjo, en0, eo0, en1, eo1, aj0, aj1);
                            if (at_i) {
                                // and at i
                                const float4 ku = nb_u[bk], kv = nb_v[bk];
                                const float cin = __builtin_fmaf(ju.z, ku.z, __builtin_fmaf(ju.y, ku.y, ju.x * ku.x));
                                const float cio = __builtin_fmaf(jv.z, kv.z, __builtin_fmaf(jv.y, kv.y, jv.x * kv.x));
                                nnp_terms<TWO>(top_p, top_m, cin, cio, en0, eo0, en1, eo1, ai0, ai1);
                            }
                        }
                    };
                    const bool writer = tg.tact && tg.part == 0;
                    if (gb >= 0) {
                        if constexpr (SPLIT) visits(std::true_type{}, std::true_type{}, tg.o0, tg.o1);
                        visits(std::true_type{}, std::false_type{}, tg.m0, tg.m1);
                        nnp_store<NP, SETS>(G1, L.gd + NNP_GD * gb, tg.lp, writer, tg.j, i, lane, Dp, s_col + set * NNP_MAXF, aj1, ai1);
                    } else {
                        if constexpr (SPLIT) visits(std::false_type{}, std::true_type{}, tg.o0, tg.o1);
                        visits(std::false_type{}, std::false_type{}, tg.m0, tg.m1);
                    }
                    nnp_store<NP, SETS>(G0, L.gd + NNP_GD * ga, tg.lp, writer, tg.j, i, lane, Dp, s_col + set * NNP_MAXF, aj0, ai0);
                }
            }
            __syncthreads();
            if constexpr (SETS > 1) {
                // the halves' sums at the moved atom, one after the other
                if (tid < T.nf) {
                    float d = Dp[tid * NP + i];
#pragma unroll
                    for (int v = 0; v < SETS; ++v) d += s_col[v * NNP_MAXF + tid];
                    Dp[tid * NP + i] = d;
                }
                __syncthreads();
            }
            nnp_forward<NP, NT>(T, L, Dp, N, L.eatn, &s_en);
            new_en = s_en;
        }
        // Metropolis, src/MCRun.jl:122-132 and src/Exchange.jl:53-57; with
        // delayed acceptance the second stage corrects the surrogate's error:
        // accept with min(1, exp(-beta ((E' - E) - (E_hat' - E_hat))))
        const double dd = new_en - E;
        bool accept;
        if (!da) {
            accept = (dd <= 0.0) || (det_exp(-dd * beta) >= (double)d0.umet);
        } else if (!stage1) {
            accept = false;
        } else {
            const u32x4 X2 = draw(a.seed, ri.run_key, RNG_MOVE, 255u, (uint32_t)t, sweep, m);
            const double x2 = dd - dEh;
            accept = (x2 <= 0.0) || (det_exp(-x2 * beta) >= (double)u24(X2.x));
        }
        if (tid == 0 && a.trace_de != nullptr && a.trace_cycle < a.trace_cycles) {
            const size_t ti = ((size_t)Tg * a.trace_cycles + a.trace_cycle) * nsteps + m;
            a.trace_de[ti] = dd;
            a.trace_acc[ti] = (int8_t)accept;
            a.trace_idx[ti] = i;
            if (da && a.trace_aux != nullptr) a.trace_aux[ti] = dEh;
        }
        if (accept) {
            // swap_atom_config! + swap_vars!(NNPVariables), src/swap_config.jl:40-51, :213-221
            float *tmp = Gp;
            Gp = Dp;
            Dp = tmp;
            for (int e = tid; e < N; e += NT) L.eat[e] = L.eatn[e];
            if (da) {
                float *t1 = Sd;
                Sd = Sn;
                Sn = t1;
                t1 = sat;
                sat = satn;
                satn = t1;
                Ehat = Ehn;
            }
            if (tid == 0) {
                L.X[i] = tx;
                L.X[NP + i] = ty;
                L.X[2 * NP + i] = tz;
            }
            E = new_en;
            nacc += 1;
        }
        __syncthreads();
    }

    // periodic full rebuild bounds the drift of the incremental features
    if (a.recompute_every > 0 && ((long long)sweep + 1) % a.recompute_every == 0) {
        nnp_full_build<NP, NT>(T, L, Gp, N);
        nnp_forward<NP, NT>(T, L, Gp, N, L.eat, &s_en);
        const double dr = __builtin_fabs(E - s_en);
        if (tid == 0 && dr > a.slot_drift[slot]) a.slot_drift[slot] = dr;
        E = s_en;
    }

    float *gX = reinterpret_cast<float *>(a.coords) + (size_t)slot * 3 * NP;
    float *gGw = a.feat + (size_t)slot * T.nf * NP;
    for (int e = tid; e < 3 * NP; e += NT) gX[e] = L.X[e];
    for (int e = tid; e < T.nf * NP; e += NT) gGw[e] = Gp[e];
    for (int e = tid; e < NP; e += NT) a.eatom[(size_t)slot * NP + e] = L.eat[e];
    if (tid == 0) {
        a.slot_en[slot] = E;
        a.t_count_atom[2 * Tg] += nacc;
        a.t_count_atom[2 * Tg + 1] += nacc;
        if (s_err) a.run_error[a.slot_run[slot]] = 1;
        if (da) {
            a.da_stats[3 * slot] += n_prop;
            a.da_stats[3 * slot + 1] += n_acc1;
            a.da_stats[3 * slot + 2] += nacc;
        }
    }
}

// Between cycles: replica exchange (src/Exchange.jl:103-155, src/MCRun.jl:203-205),
// step adaptation (src/Exchange.jl:198-263) and sampling (src/Sampling.jl:330-371),
// one wave per run: the pairs of an even/odd exchange are disjoint and go to
// lanes, and so do the temperatures.  Bound by the latency of the dependent
// reads of a pair (labels, slots, energies): one thread per run took 45 us for
// 40 temperatures, 4 so.
__global__ void __launch_bounds__(64) nnp_cycle_kernel(SweepArgs a)
{
    const RunInfo &ri = a.runs[blockIdx.x];
    const int lane = threadIdx.x;
    const int R = ri.n_temps, tb = ri.temp_base, N = ri.n_atoms;
    const uint32_t sweep = (uint32_t)a.sweep0;
    const long long pidx = a.cycle0 + 1;
    auto try_pair = [&](int n) {
        u32x4 X1 = draw(a.seed, ri.run_key, RNG_EXCH, 0u, 0u, sweep, 1u + (uint32_t)n);
        const double u = u53(X1.x, X1.y);
        const int sa = a.temp_slot[tb + n], sb = a.temp_slot[tb + n + 1];
        const double de = a.slot_en[sa] - a.slot_en[sb];
        const double db = a.t_beta[tb + n] - a.t_beta[tb + n + 1];
        double acc = det_exp(db * de);
        if (acc > 1.0) acc = 1.0;
        a.t_count_exc[2 * (tb + n)] += 1;
        a.t_count_exc[2 * (tb + n + 1)] += 1;
        if (acc > u) {
            a.t_count_exc[2 * (tb + n) + 1] += 1;
            a.t_count_exc[2 * (tb + n + 1) + 1] += 1;
            a.slot_temp[sa] = n + 1;
            a.slot_temp[sb] = n;
            a.temp_slot[tb + n] = sb;
            a.temp_slot[tb + n + 1] = sa;
        }
    };
    if (R > 1 && (sweep + 1u) % (uint32_t)a.exchange_every == 0u) {
        if (a.exchange_mode == EXC_EVEN_ODD) {
            for (int n = (int)(sweep & 1u) + 2 * lane; n + 1 < R; n += 128) try_pair(n);
        } else if (lane == 0) {
            u32x4 X0 = draw(a.seed, ri.run_key, RNG_EXCH, 0u, 0u, sweep, 0u);
            const double u = u53(X0.x, X0.y);
            if (a.exchange_mode == EXC_EVERY || u < 0.1) try_pair((int)below(X0.z, (uint32_t)(R - 1)));
        }
    }
    __syncthreads();  // the exchanged labels, before they are read by temperature
    for (int t = lane; t < R; t += 64) {
        const int T = tb + t;
        if (pidx % a.n_adjust == 0) {
            const double ar = (double)a.t_count_atom[2 * T + 1] / (double)((long long)a.n_adjust * N);
            if (ar < a.min_acc) a.t_displ[2 * T] *= 0.9;
            else if (ar > a.max_acc) a.t_displ[2 * T] *= 1.1;
            a.t_count_atom[2 * T + 1] = 0;
        }
        if (a.sampling && pidx % a.mc_sample == 0) {
            const double E = a.slot_en[a.temp_slot[T]];
            a.t_ham[2 * T] += E;
            a.t_ham[2 * T + 1] += E * E;
            const double hi = (E - ri.en_min) / ri.delta_en + 1.0;
            const int h = hi < 1.0 ? 1 : (hi > (double)a.n_bin ? a.n_bin + 2 : (int)__builtin_floor(hi) + 1);
            a.t_hist[(size_t)T * a.hist_stride + (h - 1)] += 1u;
        }
    }
}

}  // namespace ptmc
