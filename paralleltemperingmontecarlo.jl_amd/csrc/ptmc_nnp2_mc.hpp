// Monte-Carlo cycles of the two-species RuNNer potential in the NNVT
// ensemble, compiled once per element type N2R (double: FP64 throughout;
// float: binary32 positions, distances, features and networks, FP64 energy
// sums and Metropolis test) by ptmc_nnp2_mc.hip and ptmc_nnp2_mc_f32.hip.
// Reference: RuNNerPotential2Atom (src/EnergyEvaluation.jl:1287-1448,
// :1622-1643, :1748-1768, :1824-1856), NNVT (src/Ensembles.jl:138-150,
// :270-282), moves src/MCMoves.jl:115-145, :363-385, commit
// src/swap_config.jl:223-277.
//
// One workgroup owns one configuration for a cycle of N + n_swaps moves.  A
// move is an atom displacement or, with probability n_swaps / (N + n_swaps),
// an exchange of one atom of each species (slot semantics: the atoms keep
// their species and trade positions).  The trial feature matrix D is the
// current one, G, with
//   * columns of unmoved atoms: plus the change of every radial pair and
//     angular triangle holding a moved atom (new minus old, per-species scale);
//   * columns of moved atoms: rebuilt from the trial positions.
// The reference builds the same trial matrix as G plus deltas accumulated per
// pair / triangle (DeltaMatrix.jl:23-624); every sum here is formed in a fixed
// order, so a run does not depend on the schedule.
//
// The exponential and cutoffs of a triangle factor over its sides:
//   exp(-eta (r_cj^2 + r_ck^2 + r_jk^2)) f_cj f_ck f_jk = P_cj P_ck P_jk,
//   P_ab = exp(-eta r_ab^2) f_ab,
// so that a triangle costs a cosine, two products and its functions' powers,
// and exponentials are taken per pair only.  Angular functions of equal eta
// form a group with one matrix P (device memory, the slot's own, rows of 64
// lanes; read from L2, loads one partner ahead), two waves per group, each
// over every other partner k with a lane per target atom j: k's record is the
// same for all lanes, j's terms stay in registers, and the triangle's angle at
// the moved atom is summed along the way (both orders of a pair).  Powers of
// functions sorted by (lambda, zeta) come from one squaring chain.
//
// Bound by the instructions of the triangle visits (about 45 and 10 per
// function each, only partners inside the cut-off, half of a move's time) and
// the latency of the move's phases (rows, pair factors, three layers, commit):
// VALU issues in 46 % of the SIMDs' cycles, and a wave waits for 57 % of its own.
// Cu50Zn5 (5 + 26 functions, 7 groups, one workgroup of 16 waves per CU), a
// launch of 57 moves: 11.1 ms with an exponential, a division and two square
// roots per triangle and group, 1.85 ms so; 25 ladders of 10 1.35 -> 7.0e6
// moves/s, 50 ladders in binary32 2.85e6 -> 1.02e7.
// (no include guard: included once per element type)
#include "ptmc_nnp_layout.hpp"
#include "ptmc_sweep.hpp"
#include "ptmc_tanh.hpp"

namespace ptmc {

namespace {

constexpr int N2_NT = N2_THREADS;  // threads of a workgroup
constexpr int N2_NW = N2_NT / 64;
constexpr bool N2_F32 = sizeof(N2R) == 4;

// one move's draws: the atom move, and the species picks of a swap
struct N2Draw {
    MoveDraw<N2R> d;
    int p, q;
};

// The potential's tables as the kernels read them: from the kernel argument
// through a pointer that n2_fresh renews at every phase of a move, so that
// the compiler loads a field where it is used instead of keeping all of them
// (and spilling them) over the whole launch.
typedef const __attribute__((address_space(4))) SweepArgs N2Args;
typedef const __attribute__((address_space(4))) Nnp2Tables N2Tab;

__device__ __forceinline__ N2Args &n2_args()
{
    N2Args *p = (N2Args *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *p;
}
__device__ __forceinline__ N2Tab &n2_fresh() { return n2_args().nnp2; }

struct N2Group;

// LDS, most of it at offsets known to the compiler
struct N2Lds {
    N2R *rec;                     // [2][64][8]: trial position, unit vector from the moved atom's trial position
    N2Draw *dr;                   // draws of 64 moves
    struct N2Group *G;            // [pass] group records
    N2R *X;                       // [3][64] positions
    N2R *r2n, *fn, *r2o, *fo, *rin;  // [2][64] of the moved atoms: trial and old r^2 and cutoff, trial 1/r
    N2R *eat, *eatn;              // [64] per-atom energies, current and trial
    N2R *RI;                      // [N][N] inverse distances (0 on the diagonal)
    N2R *D;                       // [ng][N] trial features
    N2R *H1, *H2;                 // [h1][N], [h2][N]
    N2R *B;                       // [pass][NNP2_GMAX][2][N] changes of part 1 (over H1, H2)
    N2R *PP;                      // [2][pass][64][2]: trial and old P of the moved atoms
    N2R *S;                       // [2][n_ang][3][2] angular sums at the moved atoms
    N2R *W;                       // staged weights
};

__device__ __forceinline__ N2Lds n2_lds(N2Tab &T, int N)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    N2Lds l;
    l.rec = reinterpret_cast<N2R *>(lds_raw);
    l.dr = reinterpret_cast<N2Draw *>(l.rec + 2 * 64 * 8);
    l.G = reinterpret_cast<N2Group *>(reinterpret_cast<unsigned char *>(l.dr) + NNP2_DRAWS * NNP2_DRAW_BYTES);
    l.X = reinterpret_cast<N2R *>(reinterpret_cast<unsigned char *>(l.G) + NNP2_GP * NNP2_GROUP_BYTES);
    l.r2n = l.X + 3 * 64;
    l.fn = l.r2n + 2 * 64;
    l.r2o = l.fn + 2 * 64;
    l.fo = l.r2o + 2 * 64;
    l.rin = l.fo + 2 * 64;
    l.eat = l.rin + 2 * 64;
    l.eatn = l.eat + 64;
    l.RI = l.eatn + 64;
    l.PP = l.RI + N * N;
    l.D = l.PP + 2 * T.pass * 64 * 2;
    l.H1 = l.B = l.D + N * T.ng;
    l.H2 = l.H1 + N * T.h1;
    l.S = l.H1 + N * max(T.h1 + T.h2, 2 * NNP2_GMAX * T.pass);
    l.W = l.S + 12 * T.n_ang;
    return l;
}
static_assert(sizeof(N2Draw) <= NNP2_DRAW_BYTES, "draw record");

// type-2 cutoff 0.5 (cos(pi r / rc) + 1) (MachineLearningPotential/Cutoff.jl:79-90)
// as cos^2(pi t / 2), t = r / rc, the cosine by its Taylor series in t^2 (FP64
// through t^24, remainder below 1e-18 on [0, 1]; binary32 through t^14)
__device__ __forceinline__ N2R n2_cut(N2R r, N2R rc)
{
    constexpr int K = sizeof(N2R) == 8 ? 12 : 7;
    const N2R t = r / rc, u = t * t;
    N2R c = (N2R)cutoff_cos_coef(K);
#pragma unroll
    for (int k = K - 1; k >= 0; --k) c = fma_<N2R>(c, u, (N2R)cutoff_cos_coef(k));
    return r < rc ? c * c : N2R(0.0);
}

__device__ __forceinline__ double n2_tanh(double x)
{
    return net_tanh(x, [](double d) {
        double y = __builtin_amdgcn_rcp(d);
        y = fma(fma(-d, y, 1.0), y, y);
        return fma(fma(-d, y, 1.0), y, y);
    });
}
__device__ __forceinline__ float n2_tanh(float x) { return tanhf(x); }

__device__ __forceinline__ N2R n2_d2(const N2R *a, const N2R *b)
{
    const N2R dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
    return dx * dx + dy * dy + dz * dz;
}

// radial pair value f exp(-eta r^2), zero at f = 0 or 1 (SymmFunc.jl:229-231)
__device__ __forceinline__ N2R n2_rad(N2R r2, N2R f, N2R eta)
{
    return (f != N2R(0.0) && f != N2R(1.0)) ? f * exp(-eta * r2) : N2R(0.0);
}

// A feature's scale and offset are applied in FP64 and the feature rounded once:
// a narrow range makes both large and of opposite sign.
__device__ __forceinline__ N2R n2_scaled(N2R sum, double scale, double offset) { return (N2R)((double)sum * scale + offset); }
__device__ __forceinline__ N2R n2_changed(N2R feature, N2R change, double scale)
{
    return (N2R)((double)feature + (double)change * scale);
}

// b^zeta: integer zeta by squaring, else pow (rounding can leave b = 1 +
// lambda cos a little below zero)
__device__ __forceinline__ N2R n2_pow(N2R b, N2R zeta)
{
    if (zeta >= N2R(0.0) && zeta <= N2R(64.0) && zeta == rint(zeta)) {
        int e = (int)zeta;
        N2R r = N2R(1.0), q = b;
        while (e) {
            if (e & 1) r *= q;
            q *= q;
            e >>= 1;
        }
        return r;
    }
    return pow(zeta == rint(zeta) || b > N2R(0.0) ? b : N2R(0.0), zeta);
}

// sum over the wave, in every lane
__device__ __forceinline__ N2R n2_wave_sum(N2R v)
{
    v = group_sum<16>(v);
    v = v + row_xor<16>(v);
    return v + row_xor<32>(v);
}

__device__ __forceinline__ N2R n2_uniform(N2R v)
{
    if constexpr (sizeof(N2R) == 8) {
        const uint64_t b = (uint64_t)__double_as_longlong((double)v);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
        return (N2R)__longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
    } else {
        return (N2R)__uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint((float)v)));
    }
}

// The functions of an angular group, sorted by (lambda, zeta), uniform over
// the wave; prog[l] says how function l takes its power of b = 1 + lambda cos:
// NNP2_FRESH + n: n squarings of a new b; NNP2_CHAIN + n: n squarings of
// function l - 1's power; NNP2_POW: n2_pow (kernels compiled with POW; its
// registers would spill the visits of the others).
struct N2Group {
    N2R eta, lam[NNP2_GMAX];
    int cnt, q[NNP2_GMAX], prog[NNP2_GMAX];
};
static_assert(sizeof(N2Group) <= NNP2_GROUP_BYTES, "group record");

// records of groups g0, g0 + 1, ... of a pass into LDS
__device__ __forceinline__ void n2_stage_groups(N2Tab &T, N2Group *to, int g0)
{
    for (int u = threadIdx.x; u < T.pass * NNP2_GMAX; u += N2_NT) {
        const int gl = u / NNP2_GMAX, l = u % NNP2_GMAX;
        if (g0 + gl >= T.n_groups) continue;
        const int first = T.grp[2 * (g0 + gl)], cnt = T.grp[2 * (g0 + gl) + 1], f = first + (l < cnt ? l : 0), q = T.gfn[f];
        to[gl].cnt = cnt;
        to[gl].eta = (N2R)T.ang[(size_t)q * 15];
        to[gl].q[l] = q;
        to[gl].prog[l] = T.gprog[f];
        to[gl].lam[l] = (N2R)T.ang[(size_t)q * 15 + 1];
    }
}

// a record as uniform values
__device__ __forceinline__ void n2_load_group(const N2Group &from, N2Group &G)
{
    G.cnt = __builtin_amdgcn_readfirstlane(from.cnt);
#pragma unroll
    for (int l = 0; l < NNP2_GMAX; ++l) {
        G.q[l] = __builtin_amdgcn_readfirstlane(from.q[l]);
        G.prog[l] = __builtin_amdgcn_readfirstlane(from.prog[l]);
        G.lam[l] = n2_uniform(from.lam[l]);
    }
}

__device__ __forceinline__ N2R n2_group_eta(N2Tab &T, int g) { return (N2R)T.ang[(size_t)T.gfn[T.grp[2 * g]] * 15]; }

// powers of NC cosines for every function of the group: use(l, p)
template <bool POW, int NC, typename Use>
__device__ __forceinline__ void n2_powers(N2Tab &T, const N2Group &G, const N2R (&c)[NC], Use use)
{
    N2R b[NC];
#pragma unroll
    for (int v = 0; v < NC; ++v) b[v] = N2R(1.0);
#pragma unroll
    for (int l = 0; l < NNP2_GMAX; ++l) {
        if (l < G.cnt) {
            const int pr = G.prog[l];
            if (pr >= NNP2_FRESH) {
#pragma unroll
                for (int v = 0; v < NC; ++v) b[v] = fma_<N2R>(G.lam[l], c[v], N2R(1.0));
                asm volatile("");  // a uniform branch, not two selects per power
            }
            if (POW && pr == NNP2_POW) {
                const N2R zeta = (N2R)T.ang[(size_t)G.q[l] * 15 + 2];
#pragma unroll
                for (int v = 0; v < NC; ++v) b[v] = n2_pow(b[v], zeta);
            } else {
                for (int q = pr & 15; q > 0; --q) {
#pragma unroll
                    for (int v = 0; v < NC; ++v) b[v] *= b[v];
                }
            }
            use(l, b);
        }
    }
}

// inverse distances and the groups' P of the configuration X
__device__ __forceinline__ void n2_tables(N2R *P, int N)
{
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    for (int e = threadIdx.x; e < N * 64; e += N2_NT) {
        const int k = e >> 6, j = e & 63;
        N2R r2 = N2R(0.0), f = N2R(0.0);
        if (j < N) {
            const N2R pk[3] = {L.X[k], L.X[64 + k], L.X[128 + k]}, pj[3] = {L.X[j], L.X[64 + j], L.X[128 + j]};
            r2 = n2_d2(pk, pj);
            const N2R r = sqrt(r2);
            f = j == k ? N2R(0.0) : n2_cut(r, (N2R)T.r_cut);
            L.RI[k * N + j] = j == k ? N2R(0.0) : N2R(1.0) / r;
        }
        for (int g = 0; g < T.n_groups; ++g)
            P[((size_t)g * N + k) * 64 + j] = f != N2R(0.0) ? exp(-n2_group_eta(T, g) * r2) * f : N2R(0.0);
    }
}

// sum of terms centred on an atom over the lanes j of species 1 or 2
__device__ __forceinline__ N2R n2_species_sum(N2R v, int n1, int lane, bool second)
{
    return n2_wave_sum((lane < n1) != second ? v : N2R(0.0));
}

// a and b exchanged across bit 5 or 4 of the lane and added: lanes with the
// bit clear get a's sum over the two lanes, the others b's
template <int ROW>
__device__ __forceinline__ uint64_t n2_swap_words(uint32_t a, uint32_t b)
{
    if constexpr (ROW == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        return ((uint64_t)r[1] << 32) | r[0];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        return ((uint64_t)r[1] << 32) | r[0];
    }
}
template <int ROW>
__device__ __forceinline__ float n2_merge(float a, float b)
{
    const uint64_t r = n2_swap_words<ROW>(__float_as_uint(a), __float_as_uint(b));
    return __uint_as_float((uint32_t)r) + __uint_as_float((uint32_t)(r >> 32));
}
template <int ROW>
__device__ __forceinline__ double n2_merge(double a, double b)
{
    const uint64_t x = (uint64_t)__double_as_longlong(a), y = (uint64_t)__double_as_longlong(b);
    const uint64_t lo = n2_swap_words<ROW>((uint32_t)x, (uint32_t)y);
    const uint64_t hi = n2_swap_words<ROW>((uint32_t)(x >> 32), (uint32_t)(y >> 32));
    const uint64_t p = (hi << 32) | (uint32_t)lo, q = (hi & 0xffffffff00000000ull) | (lo >> 32);
    return __longlong_as_double((long long)p) + __longlong_as_double((long long)q);
}

// Sums of eight values over the wave: lane l gets the sum of value 4 b5 + 2 b4
// + b3 (bits of l).  The row swaps merge two values into one register per
// step, 34 instructions in place of eight butterflies' 240.
__device__ __forceinline__ N2R n2_sum8(const N2R (&v)[8], int lane)
{
    N2R a[4], b[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = n2_merge<32>(v[i], v[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i) b[i] = n2_merge<16>(a[i], a[i + 2]);
    const bool odd = (lane & 8) != 0;
    N2R s = (odd ? b[1] : b[0]) + dpp_perm<0x128>(odd ? b[0] : b[1]);  // row_ror 8: the lane across bit 3
    s = s + dpp_perm<0xB1>(s);
    s = s + dpp_perm<0x4E>(s);
    return s + dpp_perm<0x141>(s);
}

// Visits of a wave: moved atom a (the m-th), partners k = part, part + 2, ...
// of each species block, a lane per target j.  Changes of the rows of the
// wave's group at the unmoved atoms: FP64 part 0 into D, part 1 into B (added to
// D after a barrier); binary32 unscaled, part 0 kept by the wave and part 1 into B,
// for n2_add to round a row's change into D once.  Sums at the moved atom into S
// (both orders of an equal-species pair are visited).  b: the other moved atom of a swap, a
// partner at its trial position, or -1; the triangles with both moved atoms
// count at j once (m = 0).
template <bool POW, bool SWAP>
__device__ __forceinline__ void n2_visits(const N2R *Pg, int N, int gl, int m, int a, int b, int part, int lane,
                                          N2R (&kept)[2][NNP2_GMAX])
{
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    N2Group G;
    n2_load_group(L.G[gl], G);
    const int n1 = T.n1, lc = lane < N ? lane : N - 1;
    const N2R *rec = L.rec + m * 64 * 8;
    const N2R *pp = L.PP + (m * T.pass + gl) * 64 * 2;
    const N2R *po = L.PP + ((1 - m) * T.pass + gl) * 64 * 2;  // of the other moved atom
    const N2R xj = L.X[lc], yj = L.X[64 + lc], zj = L.X[128 + lc];
    const N2R pnj = lane < N ? pp[2 * lc] : N2R(0.0), poj = lane < N ? -pp[2 * lc + 1] : N2R(0.0);
    // unit vectors: trial moved atom -> j, and j -> old moved atom
    const N2R vx = rec[8 * lc + 3], vy = rec[8 * lc + 4], vz = rec[8 * lc + 5];
    const N2R rio = L.RI[a * N + lc];
    const N2R ox = (L.X[a] - xj) * rio, oy = (L.X[64 + a] - yj) * rio, oz = (L.X[128 + a] - zj) * rio;
    const bool still = lane < N && lane != a && lane != b;
    const int sc = lane < n1 ? 0 : 1, sa = a < n1 ? 0 : 1;
    // partners inside the cut-off of the trial or the old position (about two
    // thirds of a 55-atom cluster); every other one is this wave's
    uint64_t near = __ballot(lane < N && lane != a && (L.fn[m * 64 + lc] != N2R(0.0) || L.fo[m * 64 + lc] != N2R(0.0)));
    const uint64_t first = n1 >= 64 ? ~0ull : (1ull << n1) - 1ull;
    for (int blk = 0; blk < 2; ++blk) {
        uint64_t left = near & (blk ? ~first : first);
        if ((part ^ (blk ? __popcll(near & first) : 0)) & 1) left &= left - 1ull;
        N2R accJ[NNP2_GMAX], own[NNP2_GMAX];
#pragma unroll
        for (int l = 0; l < NNP2_GMAX; ++l) accJ[l] = own[l] = N2R(0.0);
        N2R pnext = left != 0ull ? Pg[__builtin_ctzll(left) * 64 + lane] : N2R(0.0);
        while (left != 0ull) {
            const int k = __builtin_ctzll(left);
            left &= left - 1ull;
            left &= left - 1ull;
            const N2R p = pnext;
            if (left != 0ull) pnext = Pg[__builtin_ctzll(left) * 64 + lane];
            const N2R *rk = rec + 8 * k;
            const N2R ri = L.RI[k * N + lc];
            const N2R wx = rk[0] - xj, wy = rk[1] - yj, wz = rk[2] - zj;
            N2R c[3];
            c[0] = -fma_<N2R>(vz, wz, fma_<N2R>(vy, wy, vx * wx)) * ri;
            c[1] = fma_<N2R>(oz, wz, fma_<N2R>(oy, wy, ox * wx)) * ri;
            c[2] = fma_<N2R>(vz, rk[5], fma_<N2R>(vy, rk[4], vx * rk[3]));
            N2R ea = p * pp[2 * k] * pnj;
            N2R en = ea, eo = p * pp[2 * k + 1] * poj;
            if constexpr (SWAP) {
                if (k == b) {
                    const N2R ux = L.X[b] - xj, uy = L.X[64 + b] - yj, uz = L.X[128 + b] - zj;
                    c[0] = -fma_<N2R>(vz, wz, fma_<N2R>(vy, wy, vx * wx)) * L.rin[(1 - m) * 64 + lc];
                    c[1] = fma_<N2R>(oz, uz, fma_<N2R>(oy, uy, ox * ux)) * ri;
                    ea = po[2 * lc] * pp[2 * k] * pnj;
                    en = m == 0 ? ea : N2R(0.0);
                    if (m != 0) eo = N2R(0.0);
                } else {
                    ea = lane == b ? po[2 * k] * pp[2 * k] * pnj : ea;
                }
            }
            n2_powers<POW, 3>(T, G, c, [&](int l, const N2R (&t)[3]) {
                accJ[l] = fma_<N2R>(eo, t[1], fma_<N2R>(en, t[0], accJ[l]));
                own[l] = fma_<N2R>(ea, t[2], own[l]);
            });
        }
        if constexpr (N2_F32) {
#pragma unroll
            for (int l = 0; l < NNP2_GMAX; ++l) {
                if (blk) kept[1][l] = accJ[l];
                else kept[0][l] = accJ[l];
                if (l < G.cnt && still && part == 1) L.B[((gl * NNP2_GMAX + l) * 2 + blk) * N + lane] = accJ[l];
            }
        } else {
            // the scales first, so that their loads are in flight together
            N2R sf[NNP2_GMAX];
#pragma unroll
            for (int l = 0; l < NNP2_GMAX; ++l) sf[l] = (N2R)T.ang[G.q[l] * 15 + 3 + 3 * sc + sa + blk];
#pragma unroll
            for (int l = 0; l < NNP2_GMAX; ++l) {
                if (l < G.cnt) {
                    const int q = G.q[l];
                    if (still) {
                        if (part == 0) L.D[(2 * T.n_rad + 3 * q + sa + blk) * N + lane] += accJ[l] * sf[l];
                        else L.B[((gl * NNP2_GMAX + l) * 2 + blk) * N + lane] = accJ[l] * sf[l];
                    }
                }
            }
        }
        for (int sj = 0; sj <= blk; ++sj) {  // j of species 1, then of species 2 with k of species 2
            N2R v[8] = {N2R(0.0), N2R(0.0), N2R(0.0), N2R(0.0), N2R(0.0), N2R(0.0), N2R(0.0), N2R(0.0)};
#pragma unroll
            for (int l = 0; l < NNP2_GMAX; ++l) v[l] = (lane < n1) == (sj == 0) ? own[l] : N2R(0.0);
            const N2R sum = n2_sum8(v, lane);
            const int l = (lane >> 5) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1);
            if ((lane & 7) == 0 && l < G.cnt)
                L.S[((m * T.n_ang + L.G[gl].q[l]) * 3 + blk + sj) * 2 + part] = blk == sj ? N2R(0.5) * sum : sum;
        }
    }
}
static_assert(NNP2_GMAX <= 8, "n2_sum8 covers a group");

__device__ __forceinline__ N2R n2_act(int code, N2R s) { return code == 2 ? n2_tanh(s) : s; }

typedef N2R n2_x4 __attribute__((ext_vector_type(4)));
typedef double n2_d4 __attribute__((ext_vector_type(4)));
typedef float n2_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ n2_d4 n2_mfma(double a, double b, n2_d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ n2_f4 n2_mfma(float a, float b, n2_f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// One hidden layer of all atoms, out[h][N] = act(in[n][N] W + b), as 16 x 16
// tiles (atoms x outputs) on the matrix cores: a wave per (species, tile) that
// holds atoms of the species, whose rows it keeps.  Lane l holds A[row l % 16]
// [k l / 16], B[k l / 16][column l % 16]; of the product value v belongs to
// row 4 v + l / 16 (FP64) or 4 (l / 16) + v (binary32).  The weights come from
// LDS where they were staged, else from L2, eight steps of k in flight.  The
// activations follow over all threads: a tile's own lanes would spend the
// padding's share on tanh too (20 outputs of 32).
// lw: the layer's weights in LDS per species, or -1.
__device__ __forceinline__ void n2_layer(const N2R *in, N2R *out, int N, int n, int h, int o, int act, const N2R *Wl,
                                         int lw0, int lw1)
{
    N2Tab &T = n2_fresh();
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lk = lane >> 4, n1 = T.n1;
    // tiles of species 1 (atoms 0 .. n1 - 1), then of species 2
    const int nct = (h + 15) / 16, nt1 = (n1 + 15) / 16 * nct, r2 = n1 / 16;
    const int nt = nt1 + (n1 < N ? ((N + 15) / 16 - r2) * nct : 0);
    for (int task = w; task < nt; task += N2_NW) {
        const bool s = task >= nt1;
        const int tt = s ? task - nt1 : task, rt = tt / nct + (s ? r2 : 0), ct = tt % nct;
        const int lo = s ? n1 : 0, hi = s ? N : n1, lw = s ? lw1 : lw0;
        const double *W = (s ? T.p2 : T.p1) + o;
        const int at = min(16 * rt + lr, N - 1), j = min(16 * ct + lr, h - 1);
        n2_x4 acc = {N2R(0.0), N2R(0.0), N2R(0.0), N2R(0.0)};
        auto steps = [&](auto weight) {
            const N2R *xp = in + lk * N + at;
            int e = lk * h + j, k0 = 0;
            for (; k0 + 32 <= n; k0 += 32, xp += 32 * N, e += 32 * h) {
                N2R x[8], y[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    y[u] = weight(e + 4 * u * h);
                    x[u] = xp[4 * u * N];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) acc = n2_mfma(x[u], y[u], acc);
            }
            for (; k0 < n; k0 += 4, xp += 4 * N, e += 4 * h) {
                const bool in_row = k0 + lk < n;
                const N2R y = weight(in_row ? e : j), x = in_row ? *xp : N2R(0.0);
                acc = n2_mfma(x, y, acc);
            }
        };
        if (lw >= 0) steps([&](int e) { return Wl[lw + e]; });
        else steps([&](int e) { return (N2R)W[e]; });
        if (16 * ct + lr < h) {
            const N2R bias = lw >= 0 ? Wl[lw + n * h + j] : (N2R)W[n * h + j];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * rt + (sizeof(N2R) == 8 ? 4 * v + lk : 4 * lk + v);
                if (row >= lo && row < hi) out[j * N + row] = acc[v] + bias;
            }
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < h * N; e += N2_NT) out[e] = n2_act(act, out[e]);
    __syncthreads();
}

// per-atom energies of D into eatn (RuNNer layout: per layer the input-major
// weights, then the biases; one network per species); returns the FP64 total
// in wave 0
__device__ __forceinline__ double n2_forward(int N)
{
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    const int tid = threadIdx.x, lane = tid & 63, ng = T.ng, h1 = T.h1, h2 = T.h2;
    // LDS holds (as T.stage says) layers 2 and 3 of both species, then layer 1
    // of species 1, or of species 1 and 2
    const int o2 = ng * h1 + h1, n23 = h1 * h2 + h2 + h2 + 1, st = T.stage;
    n2_layer(L.D, L.H1, N, ng, h1, 0, T.act1, L.W, st > 1 ? 2 * n23 : -1, st > 2 ? 2 * n23 + o2 : -1);
    n2_layer(L.H1, L.H2, N, h1, h2, o2, T.act2, L.W, st > 0 ? 0 : -1, st > 0 ? n23 : -1);
    double tot = 0.0;
    if (tid < 64) {
        const int lc = lane < N ? lane : N - 1;
        auto output = [&](auto weight) {
            N2R s = N2R(0.0);
#pragma unroll 8
            for (int k = 0; k < h2; ++k) s = fma_<N2R>(L.H2[k * N + lc], weight(k), s);
            return s + weight(h2);
        };
        N2R y;
        if (st > 0) {
            const N2R *p = L.W + (lc < T.n1 ? 0 : n23) + h1 * h2 + h2;
            y = output([&](int k) { return p[k]; });
        } else {
            const double *p = (lc < T.n1 ? T.p1 : T.p2) + o2 + h1 * h2 + h2;
            y = output([&](int k) { return (N2R)p[k]; });
        }
        y = n2_act(T.act3, y);
        if (lane < N) {
            L.eatn[lane] = y;
            tot = (double)y;
        }
        tot = group_sum<16>(tot);
        tot = tot + row_xor<16>(tot);
        tot = tot + row_xor<32>(tot);
    }
    return tot;
}

// every column rebuilt from X: P, RI, D, eatn and the total
template <bool POW>
__device__ __forceinline__ double n2_rebuild(N2R *P, int N, double *s_tot)
{
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n1 = T.n1, lc = lane < N ? lane : N - 1;
    __syncthreads();
    n2_tables(P, N);
    for (int g0 = 0; g0 == 0 || g0 < T.n_groups; g0 += T.pass) {
        n2_stage_groups(T, L.G, g0);
        __syncthreads();
        // columns x (groups of the pass, then the radial functions)
        const int ngp = min(T.pass, T.n_groups - g0);
        for (int u = w; u < N * (ngp + (g0 == 0 ? T.n_rad : 0)); u += N2_NW) {
            const int c = u % N, gl = u / N, g = g0 + gl, sc = c < n1 ? 0 : 1;
            const N2R x = L.X[c], y = L.X[64 + c], z = L.X[128 + c];
            if (gl >= ngp) {
                const int q = gl - ngp;
                const double *R = T.rad + (size_t)q * 9;
                const N2R pc[3] = {x, y, z}, pj[3] = {L.X[lc], L.X[64 + lc], L.X[128 + lc]};
                const N2R r2 = n2_d2(pc, pj);
                const N2R v = lane < N && lane != c ? n2_rad(r2, n2_cut(sqrt(r2), (N2R)T.r_cut), (N2R)R[0]) : N2R(0.0);
                for (int r = 0; r < 2; ++r) {
                    const N2R s = n2_wave_sum((lane < n1) == (r == 0) ? v : N2R(0.0));
                    if (lane == 0) L.D[(size_t)(2 * q + r) * N + c] = n2_scaled(s, R[1 + 2 * sc + r], R[5 + 2 * sc + r]);
                }
                continue;
            }
            N2Group G;
            n2_load_group(L.G[gl], G);
            const N2R *Pg = P + (size_t)g * N * 64;
            const N2R rj = L.RI[c * N + lc], pj = lane < N ? Pg[(size_t)c * 64 + lane] : N2R(0.0);
            const N2R vx = (L.X[lc] - x) * rj, vy = (L.X[64 + lc] - y) * rj, vz = (L.X[128 + lc] - z) * rj;
            for (int blk = 0; blk < 2; ++blk) {
                N2R own[NNP2_GMAX];
#pragma unroll
                for (int l = 0; l < NNP2_GMAX; ++l) own[l] = N2R(0.0);
                for (int k = blk ? n1 : 0; k < (blk ? N : n1); ++k) {
                    const N2R e = Pg[(size_t)k * 64 + lane] * Pg[(size_t)c * 64 + k] * pj, rk = L.RI[c * N + k];
                    const N2R wx = (L.X[k] - x) * rk, wy = (L.X[64 + k] - y) * rk, wz = (L.X[128 + k] - z) * rk;
                    const N2R cs[1] = {fma_<N2R>(vz, wz, fma_<N2R>(vy, wy, vx * wx))};
                    n2_powers<POW, 1>(T, G, cs, [&](int l, const N2R (&t)[1]) { own[l] = fma_<N2R>(e, t[0], own[l]); });
                }
#pragma unroll
                for (int l = 0; l < NNP2_GMAX; ++l) {
                    if (l < G.cnt) {
                        const int q = G.q[l];
                        auto store = [&](int row, N2R v) {
                            const double *A = T.ang + (size_t)q * 15 + 3 * sc + row;
                            if (lane == 0) L.D[(size_t)(2 * T.n_rad + 3 * q + row) * N + c] = n2_scaled(v, A[3], A[9]);
                        };
                        // both orders of an equal-species pair were visited
                        const N2R v = n2_species_sum(own[l], n1, lane, false);
                        store(blk, blk ? v : N2R(0.5) * v);
                        if (blk) store(2, N2R(0.5) * n2_species_sum(own[l], n1, lane, true));
                    }
                }
            }
        }
        __syncthreads();
    }
    const double tot = n2_forward(N);
    if (threadIdx.x == 0) *s_tot = tot;
    __syncthreads();
    return *s_tot;
}

__device__ __forceinline__ void n2_load_x(N2Args &a, const N2Lds &L, int slot, int N)
{
    const N2R *gX = reinterpret_cast<const N2R *>(a.coords) + (size_t)slot * 3 * NNP_NP;
    for (int e = threadIdx.x; e < 3 * N; e += N2_NT) L.X[(e / N) * 64 + e % N] = gX[(e / N) * NNP_NP + e % N];
}

// the weights T.stage says, once per launch
__device__ __forceinline__ void n2_stage_weights(N2Tab &T, N2R *W)
{
    const int o2 = T.ng * T.h1 + T.h1, n23 = T.h1 * T.h2 + T.h2 + T.h2 + 1;
    if (T.stage > 0)
        for (int e = threadIdx.x; e < 2 * n23; e += N2_NT) W[e] = (N2R)(e < n23 ? T.p1[o2 + e] : T.p2[o2 + e - n23]);
    for (int s = 0; s + 2 <= T.stage; ++s)
        for (int e = threadIdx.x; e < o2; e += N2_NT) W[2 * n23 + s * o2 + e] = (N2R)(s ? T.p2 : T.p1)[e];
}

__device__ __forceinline__ N2R *n2_pairs(N2Tab &T, int slot, int N)
{
    return reinterpret_cast<N2R *>(T.pair) + (size_t)slot * T.n_groups * N * 64;
}

// set_variables + initialise_energy (src/EnergyEvaluation.jl:1824-1856, :1748-1768)
template <bool POW>
__global__ void __launch_bounds__(N2_NT) nnp2_init_kernel(SweepArgs)
{
    N2Args &a = n2_args();
    __shared__ double s_tot;
    const int slot = blockIdx.x;
    if (a.init_run >= 0 && a.slot_run[slot] != a.init_run) return;  // whole workgroup
    N2Tab &T = a.nnp2;
    const int N = a.runs[a.slot_run[slot]].n_atoms;
    const N2Lds L = n2_lds(T, N);
    n2_load_x(a, L, slot, N);
    n2_stage_weights(T, L.W);
    const double E = n2_rebuild<POW>( n2_pairs(T, slot, N), N, &s_tot);
    N2R *gG = reinterpret_cast<N2R *>(T.feat) + (size_t)slot * NNP_NP * T.ng;
    for (int e = threadIdx.x; e < N * T.ng; e += N2_NT) gG[e] = L.D[e];
    for (int e = threadIdx.x; e < NNP_NP; e += N2_NT)
        reinterpret_cast<N2R *>(T.eatom)[(size_t)slot * NNP_NP + e] = e < N ? L.eatn[e] : N2R(0.0);
    if (threadIdx.x == 0) a.slot_en[slot] = E;
}

// the moved atoms of a move (b = -1: one) and the trial position of one
struct N2Move {
    int a, b;
    bool swap;
    N2R tr[3];
    __device__ int atom(int m) const { return m ? b : a; }
    __device__ int other(int m) const { return m ? a : b; }
};

// Rows of the moved atoms: distances, cutoffs and unit vectors in the trial
// configuration (waves 0, 1), distances and cutoffs in the old one (waves 2, 3).
__device__ __forceinline__ void n2_rows(const N2Lds &L, const N2Move &mv, int N, int w, int lane, N2R rcut)
{
    const int mm = w & 1, aa = mv.atom(mm);
    if (w >= 4 || (mm && !mv.swap) || lane >= N) return;
    auto pos = [&](int j, N2R (&x)[3]) {
        const bool now = w < 2;
        const int i = now && mv.swap ? (j == mv.a ? mv.b : (j == mv.b ? mv.a : j)) : j;
        const bool moved = now && !mv.swap && j == mv.a;
        for (int k = 0; k < 3; ++k) x[k] = moved ? mv.tr[k] : L.X[64 * k + i];
    };
    N2R xa[3], xj[3];
    pos(aa, xa);
    pos(lane, xj);
    const N2R r2 = lane == aa ? N2R(0.0) : n2_d2(xa, xj);
    const N2R r = sqrt(r2), f = n2_cut(r, rcut);
    if (w < 2) {
        const N2R iv = lane == aa ? N2R(0.0) : N2R(1.0) / r;
        L.r2n[mm * 64 + lane] = r2;
        L.fn[mm * 64 + lane] = f;
        L.rin[mm * 64 + lane] = iv;
        N2R *rk = L.rec + (mm * 64 + lane) * 8;
        for (int k = 0; k < 3; ++k) {
            rk[k] = xj[k];
            rk[3 + k] = (xj[k] - xa[k]) * iv;
        }
    } else {
        L.r2o[mm * 64 + lane] = r2;
        L.fo[mm * 64 + lane] = f;
    }
}

// trial P of atom aa (the mm-th moved one) at eta, lane j; zero at itself
__device__ __forceinline__ N2R n2_trial_pair(const N2Lds &L, N2R eta, int mm, int aa, int lane)
{
    const N2R f = L.fn[mm * 64 + lane];
    return lane != aa && f != N2R(0.0) ? exp(-eta * L.r2n[mm * 64 + lane]) * f : N2R(0.0);
}

// Radial rows of moved atom mm, function q by the wave: changes at the
// unmoved atoms, rebuilt entries at the moved one.
__device__ __forceinline__ void n2_radial(int q, const N2Move &mv, int mm, int N, int lane)
{
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    const int n1 = T.n1, lc = lane < N ? lane : N - 1, aa = mv.atom(mm), sa = aa < n1 ? 0 : 1, sc = lane < n1 ? 0 : 1;
    const double *R = T.rad + (size_t)q * 9;
    const N2R eta = (N2R)R[0];
    const N2R vn = lane < N ? n2_rad(L.r2n[mm * 64 + lc], L.fn[mm * 64 + lc], eta) : N2R(0.0);
    if (lane < N && lane != mv.a && lane != mv.b) {
        const N2R vo = n2_rad(L.r2o[mm * 64 + lc], L.fo[mm * 64 + lc], eta);
        N2R &d = L.D[(2 * q + sa) * N + lane];
        d = n2_changed(d, vn - vo, R[1 + 2 * sc + sa]);
    }
    for (int r = 0; r < 2; ++r) {
        const N2R v = n2_species_sum(vn, n1, lane, r == 1);
        if (lane == 0) L.D[(2 * q + r) * N + aa] = n2_scaled(v, R[1 + 2 * sa + r], R[5 + 2 * sa + r]);
    }
}

// Binary32: both parts' changes of the wave's group at an unmoved atom into D.
__device__ __forceinline__ void n2_add(const N2Lds &L, N2Tab &T, const N2R (&kept)[2][NNP2_GMAX], int N, int gl, int sa,
                                       int lane)
{
    const int sc = lane < T.n1 ? 0 : 1, cnt = __builtin_amdgcn_readfirstlane(L.G[gl].cnt);
#pragma unroll
    for (int l = 0; l < NNP2_GMAX; ++l) {
        if (l < cnt) {
            const int q = __builtin_amdgcn_readfirstlane(L.G[gl].q[l]);
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                N2R &d = L.D[(2 * T.n_rad + 3 * q + sa + blk) * N + lane];
                d = n2_changed(d, kept[blk][l] + L.B[((gl * NNP2_GMAX + l) * 2 + blk) * N + lane],
                               T.ang[q * 15 + 3 + 3 * sc + sa + blk]);
            }
        }
    }
}

// Angular and radial rows of the trial features: the groups T.pass at a
// time, two waves each; all threads call.
template <bool POW>
__device__ __forceinline__ void n2_features(const N2Move &mv, N2R *P, int N, int w, int lane)
{
    const int nm = mv.swap ? 2 : 1, gl = w >> 1, part = w & 1;
    for (int g0 = 0; g0 == 0 || g0 < n2_fresh().n_groups; g0 += n2_fresh().pass) {
        const int ngp = min(n2_fresh().pass, n2_fresh().n_groups - g0);
        if (g0 > 0) __syncthreads();
        {
            // P of the moved atoms, trial and old
            N2Tab &T = n2_fresh();
            const N2Lds L = n2_lds(T, N);
            if (T.n_groups > T.pass) n2_stage_groups(T, L.G, g0);
            if (T.n_groups > T.pass) __syncthreads();
            for (int u = w; u < nm * ngp; u += N2_NW) {
                const int mm = u >= ngp, g = mm ? u - ngp : u, aa = mv.atom(mm);
                if (lane < N) {
                    N2R *pp = L.PP + ((mm * T.pass + g) * 64 + lane) * 2;
                    const N2R old = P[((size_t)(g0 + g) * N + aa) * 64 + lane];
                    pp[0] = n2_trial_pair(L, L.G[g].eta, mm, aa, lane);
                    pp[1] = old;
                }
            }
        }
        __syncthreads();
        for (int mm = 0; mm < nm; ++mm) {
            const int aa = mv.atom(mm);
            N2R kept[2][NNP2_GMAX];
            if (gl < ngp) {
                const N2R *Pg = P + (size_t)(g0 + gl) * N * 64;
                if (mv.swap) n2_visits<POW, true>(Pg, N, gl, mm, aa, mv.other(mm), part, lane, kept);
                else n2_visits<POW, false>(Pg, N, gl, mm, aa, -1, part, lane, kept);
            }
            // radial functions, by the waves without a group if there are any
            const int idle = N2_NW - 2 * ngp;
            if (g0 == 0 && (idle == 0 || w >= 2 * ngp))
                for (int q = idle ? w - 2 * ngp : w; q < n2_fresh().n_rad; q += idle ? idle : N2_NW)
                    n2_radial(q, mv, mm, N, lane);
            __syncthreads();
            N2Tab &T = n2_fresh();
            const N2Lds L = n2_lds(T, N);
            const int sa = aa < T.n1 ? 0 : 1;
            if constexpr (N2_F32) {
                if (gl < ngp && part == 0 && lane < N && lane != mv.a && lane != mv.b) n2_add(L, T, kept, N, gl, sa, lane);
            } else {
                for (int u = w; u < ngp * 2 * NNP2_GMAX; u += N2_NW) {
                    const int g = u / (2 * NNP2_GMAX), l = u % (2 * NNP2_GMAX) / 2, blk = u & 1;
                    if (l < L.G[g].cnt && lane < N && lane != mv.a && lane != mv.b)
                        L.D[(2 * T.n_rad + 3 * L.G[g].q[l] + sa + blk) * N + lane] += L.B[u * N + lane];
                }
            }
            if (mm + 1 < nm) __syncthreads();
        }
    }
    __syncthreads();
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    for (int u = threadIdx.x; u < nm * T.n_ang * 3; u += N2_NT) {
        const int mm = u >= T.n_ang * 3, v = mm ? u - T.n_ang * 3 : u, q = v / 3, row = v % 3, aa = mv.atom(mm);
        const double *A = T.ang + (size_t)q * 15 + 3 * (aa < T.n1 ? 0 : 1) + row;
        L.D[(2 * T.n_rad + 3 * q + row) * N + aa] = n2_scaled(L.S[2 * u] + L.S[2 * u + 1], A[3], A[9]);
    }
    __syncthreads();
}

// An accepted move: positions, distances, pair factors, features, energies
// (swap_atom_config! / swap_move_config! with swap_vars!(NNPVariables2a)).
__device__ __forceinline__ void n2_commit(const N2Move &mv, N2R *P, N2R *gG, int N, int w, int lane)
{
    N2Tab &T = n2_fresh();
    const N2Lds L = n2_lds(T, N);
    const int nm = mv.swap ? 2 : 1, tid = threadIdx.x;
    if (w < nm && lane < N) {
        const int aa = mv.atom(w);
        const N2R v = L.rin[w * 64 + lane];
        L.RI[aa * N + lane] = v;
        L.RI[lane * N + aa] = v;
    }
    for (int u = w; u < nm * T.n_groups; u += N2_NW) {
        const int mm = u >= T.n_groups, g = mm ? u - T.n_groups : u, aa = mv.atom(mm);
        if (lane < N) {
            const N2R v = T.n_groups <= T.pass ? L.PP[((mm * T.pass + g) * 64 + lane) * 2]
                                               : n2_trial_pair(L, n2_group_eta(T, g), mm, aa, lane);
            P[((size_t)g * N + aa) * 64 + lane] = v;
            P[((size_t)g * N + lane) * 64 + aa] = v;
        }
    }
    for (int e = tid; e < N * T.ng; e += N2_NT) gG[e] = L.D[e];
    if (tid < 3 * nm) {
        const int mm = tid >= 3, k = mm ? tid - 3 : tid, aa = mv.atom(mm);
        L.X[k * 64 + aa] = L.rec[(mm * 64 + aa) * 8 + k];
    }
    if (tid < N) L.eat[tid] = L.eatn[tid];
}

// One cycle (N + n_swaps moves) of one configuration per workgroup
// (mc_step! / mc_move!, src/MCRun.jl:142-182, with get_energy!(NNVT) :87-112).
template <bool POW>
__global__ void __launch_bounds__(N2_NT) nnp2_sweep_kernel(SweepArgs)
{
    __shared__ int s_err, s_acc;
    __shared__ double s_en;
    const int slot = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    N2Args &a = n2_args();
    const RunInfo &ri = a.runs[a.slot_run[slot]];
    const int N = __builtin_amdgcn_readfirstlane(ri.n_atoms);
    const uint32_t nsteps = (uint32_t)(N + a.nnp2.n_swaps), sweep = (uint32_t)a.sweep0;
    const uint32_t run_key = __builtin_amdgcn_readfirstlane(ri.run_key);
    const int t = __builtin_amdgcn_readfirstlane(a.slot_temp[slot]);
    const int Tg = __builtin_amdgcn_readfirstlane(ri.temp_base + t);
    const double beta = a.t_beta[Tg];
    const N2R delta_r = n2_uniform((N2R)a.t_displ[2 * Tg]), radius2 = n2_uniform((N2R)ri.radius2);
    N2R *gG = reinterpret_cast<N2R *>(a.nnp2.feat) + (size_t)slot * NNP_NP * a.nnp2.ng;  // [ng][N]
    N2R *P = n2_pairs(a.nnp2, slot, N);
    {
        const N2Lds L = n2_lds(a.nnp2, N);
        n2_load_x(a, L, slot, N);
        n2_stage_groups(a.nnp2, L.G, 0);
        n2_stage_weights(a.nnp2, L.W);
        if (tid < N) L.eat[tid] = reinterpret_cast<const N2R *>(a.nnp2.eatom)[(size_t)slot * NNP_NP + tid];
        if (tid == 0) {
            s_err = 0;
            s_en = a.slot_en[slot];
        }
    }
    __syncthreads();
    n2_tables(P, N);
    double E = s_en;
    int nacc = 0, nsw = 0, nsw_acc = 0;

    for (uint32_t m = 0; m < nsteps; ++m) {
        N2Move mv;
        {
            N2Args &a = n2_args();
            N2Tab &T = a.nnp2;
            const N2Lds L = n2_lds(T, N);
            // the draws of 64 moves at a time, one lane each: the move index as
            // mc_move! draws it (src/MCRun.jl:145), a trial displacement and the
            // atoms of a swap (src/MCMoves.jl:363-370)
            if (m % NNP2_DRAWS == 0) {
                if (tid < NNP2_DRAWS && m + tid < nsteps) {
                    N2Draw r;
                    r.d = move_draw<N2R>(a.seed, run_key, (uint32_t)t, sweep, m + tid, 0u, nsteps);
                    r.p = r.q = 0;
                    if (r.d.index >= (uint32_t)N) {
                        const u32x4 S = draw(a.seed, run_key, RNG_MOVE, 254u, (uint32_t)t, sweep, m + tid);
                        r.p = (int)below(S.x, (uint32_t)T.n1);
                        r.q = T.n1 + (int)below(S.y, (uint32_t)(N - T.n1));
                    }
                    L.dr[tid] = r;
                }
                __syncthreads();
            }
            const N2Draw &dr = L.dr[m % NNP2_DRAWS];
            mv.swap = __builtin_amdgcn_readfirstlane((int)(dr.d.index >= (uint32_t)N)) != 0;
            mv.a = __builtin_amdgcn_readfirstlane(mv.swap ? dr.p : (int)dr.d.index);
            mv.b = __builtin_amdgcn_readfirstlane(mv.swap ? dr.q : -1);
            mv.tr[0] = mv.tr[1] = mv.tr[2] = N2R(0.0);
            if (!mv.swap) {
                // trial position (src/MCMoves.jl:115-135), every thread the same
                const int i = mv.a;
                make_trial<N2R, BC_SPHERE, false>(L.X[i], L.X[64 + i], L.X[128 + i], dr.d, delta_r, N2R(0.0), N2R(0.0),
                                                  mv.tr[0], mv.tr[1], mv.tr[2]);
                int count = 0;
                uint32_t attempt = 0;
                while (outside_sphere<N2R>(mv.tr[0], mv.tr[1], mv.tr[2], radius2)) {
                    count += 1;
                    if (count == 50) {
                        // recentre! (src/Configurations.jl:79-85)
                        __syncthreads();
                        if (tid < 3) {
                            double cm = 0.0;
                            for (int b = 0; b < N; ++b) cm += L.X[tid * 64 + b];
                            cm /= (double)N;
                            for (int b = 0; b < N; ++b) L.X[tid * 64 + b] = (N2R)((double)L.X[tid * 64 + b] - cm);
                        }
                        __syncthreads();
                    } else {
                        attempt += 1;
                        const MoveDraw<N2R> dd = move_draw<N2R>(a.seed, run_key, (uint32_t)t, sweep, m, attempt, nsteps);
                        make_trial<N2R, BC_SPHERE, false>(L.X[i], L.X[64 + i], L.X[128 + i], dd, delta_r, N2R(0.0),
                                                          N2R(0.0), mv.tr[0], mv.tr[1], mv.tr[2]);
                        if (count == 100) {
                            if (tid == 0) s_err = 1;
                            break;
                        }
                    }
                }
            }
            // D = G, eight loads in flight over the rows of the moved atoms
            const int nd = N * T.ng;
            N2R g[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) g[u] = gG[min(tid + u * N2_NT, nd - 1)];
            n2_rows(L, mv, N, w, lane, (N2R)T.r_cut);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (tid + u * N2_NT < nd) L.D[tid + u * N2_NT] = g[u];
            for (int e = tid + 8 * N2_NT; e < nd; e += N2_NT) L.D[e] = gG[e];
        }
        __syncthreads();
        n2_features<POW>(mv, P, N, w, lane);
        const double new_en = n2_forward(N);
        // Metropolis on the energy change (src/Exchange.jl:53-57, :74-83), by wave 0
        if (w == 0) {
            N2Args &a = n2_args();
            const N2Lds L = n2_lds(a.nnp2, N);
            const double dd = new_en - E;
            const bool ok = (dd <= 0.0) || (det_exp(-dd * beta) >= L.dr[m % NNP2_DRAWS].d.umet);
            if (tid == 0) {
                s_acc = ok;
                s_en = new_en;
                if (a.trace_de != nullptr && a.trace_cycle < a.trace_cycles) {
                    const size_t ti = ((size_t)Tg * a.trace_cycles + a.trace_cycle) * nsteps + m;
                    a.trace_de[ti] = dd;
                    a.trace_acc[ti] = (int8_t)ok;
                    a.trace_idx[ti] = mv.swap ? N + mv.a * N + mv.b : mv.a;
                }
            }
        }
        __syncthreads();
        if (mv.swap) nsw += 1;
        if (__builtin_amdgcn_readfirstlane(s_acc)) {
            n2_commit(mv, P, gG, N, w, lane);
            E = s_en;
            if (mv.swap) nsw_acc += 1;
            else nacc += 1;
        }
        __syncthreads();
    }

    N2Args &z = n2_args();
    const N2Lds L = n2_lds(z.nnp2, N);
    // periodic full rebuild bounds the drift of the incremental features
    if (z.recompute_every > 0 && ((long long)sweep + 1) % z.recompute_every == 0) {
        __shared__ double s_tot;
        const double Er = n2_rebuild<POW>(P, N, &s_tot);
        const double dr = __builtin_fabs(E - Er);
        if (tid == 0 && dr > z.slot_drift[slot]) z.slot_drift[slot] = dr;
        for (int e = tid; e < N * z.nnp2.ng; e += N2_NT) gG[e] = L.D[e];
        if (tid < N) L.eat[tid] = L.eatn[tid];
        E = Er;
        __syncthreads();
    }

    N2R *gX = reinterpret_cast<N2R *>(z.coords) + (size_t)slot * 3 * NNP_NP;
    for (int e = tid; e < 3 * N; e += N2_NT) gX[(e / N) * NNP_NP + e % N] = L.X[(e / N) * 64 + e % N];
    if (tid < N) reinterpret_cast<N2R *>(z.nnp2.eatom)[(size_t)slot * NNP_NP + tid] = L.eat[tid];
    if (tid == 0) {
        z.slot_en[slot] = E;
        z.t_count_atom[2 * Tg] += nacc;
        z.t_count_atom[2 * Tg + 1] += nacc;
        z.t_count_vol[2 * Tg] += nsw_acc;
        z.t_count_vol[2 * Tg + 1] += nsw;
        if (s_err) z.run_error[z.slot_run[slot]] = 1;
    }
}

}  // namespace

using SweepFn = void (*)(SweepArgs);

SweepFn N2_SWEEP_FN(bool pow) { return pow ? &nnp2_sweep_kernel<true> : &nnp2_sweep_kernel<false>; }
SweepFn N2_INIT_FN(bool pow) { return pow ? &nnp2_init_kernel<true> : &nnp2_init_kernel<false>; }

}  // namespace ptmc
