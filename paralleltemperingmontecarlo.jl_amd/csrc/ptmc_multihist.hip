// Multihistogram heat capacities (multihistogram_NVT, src/multihist_NVT.jl:11-221,
// and multihistogram_NPT, src/multihist_NPT.jl:17-340) in FP64 on the device.
//
// The reference iterates free energies f_i = log sum_m q(beta_i, m) with
//   q(b, m) = H_m / D_m * exp(-b h_m - off_m),
//   off_m   = max(-1e6, max_i(-beta_i h_m - f_i)) + log(1000),
//   D_m     = sum_i n_i exp(-beta_i h_m - f_i - off_m),  H_m = sum_i h_i(m),
// over the energy bins (h = E), or the (energy, volume) bins with h = E + pV.
// off_m cancels from q, so it may be taken from any earlier free energies f0:
// with K_im = exp(-beta_i h_m - f0_i - off_m(f0)) an iteration is
//   D_m = sum_i n_i K_im exp(-(f_i - f0_i)),  f_i = f0_i + log sum_m H_m K_im / D_m,
// two products with a matrix that stays, and no exponential per (i, m).  K is
// rebuilt (f0 = f) once some |f_i - f0_i| passes MH_REBASE, long before a
// term that matters could leave the range of a double.  Heat capacities
// follow on the output grid: C = (<h^2> - <h>^2) / (k T^2).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/ptmc.h"
#include "ptmc_device.hpp"
#include "ptmc_multihist_cut.hpp"

using namespace ptmc;

namespace {

constexpr double MH_REBASE = 16.0;
constexpr unsigned MH_SPIN = 1u << 26;         // polls of a grid barrier before it gives up (seconds)

struct MHArgs {
    int n_temps, n_bin, n_bins, n_res, max_iter;  // n_bins: n_bin (NVT) or n_bin^2 (NPT) bins of a run
    int npt, n_wg, n_blk, wg_blk;  // workgroups of a run, its blocks of MH_BINS bins, blocks of a workgroup
    double conv;
    const double *beta;      // runs x R
    const double *hist;      // runs x R x (n_bin + 2), or x (n_bin + 2)^2: rows energy, columns volume
    const double *en_min, *en_max, *v_min, *v_max, *pressure;  // runs
    const double *beta_res;  // runs x n_res
    const double *t_res;     // runs x n_res
    double k_boltzmann;
    double *c;               // runs x n_res heat capacities
    double *moments;         // runs x n_res x 3: <E>, <V>, <h>, or null
    double *free_energy;     // runs x R, or null
    int *iterations;         // runs, or null
    double *ncyc;            // runs x R histogram totals, or null: each workgroup forms its run's
    double *off, *ratio;     // runs x n_bins: offsets and H_m / D_m of the last free energies
    double *hsum;            // runs x n_bins histogram sums H_m (slices that are not kept)
    double *part;            // runs x 2 x n_blk x R block sums (n_wg > 1)
    unsigned *count;         // runs arrivals at the barrier, zeroed (n_wg > 1)
    int *error;              // set when a barrier gave up, zeroed (n_wg > 1)
};

// energy and volume of bin b, from the run's range
struct MHBins {
    int nb, npt;
    double emin, de, vmin, dv, p;
    __device__ MHBins(const MHArgs &a, int run) : nb(a.n_bin), npt(a.npt)
    {
        emin = a.en_min[run];
        de = (a.en_max[run] - emin) / (double)nb;
        vmin = dv = p = 0.0;
        if (npt) {
            vmin = a.v_min[run];
            dv = (a.v_max[run] - vmin) / (double)nb;
            p = a.pressure[run];
        }
    }
    __device__ double energy(int b) const { return emin + ((double)((npt ? b / nb : b) + 1) - 0.5) * de; }
    __device__ double volume(int b) const { return npt ? vmin + ((double)(b % nb + 1) - 0.5) * dv : 0.0; }
    __device__ double h(int b) const { return npt ? energy(b) + p * volume(b) : energy(b); }
    __device__ size_t stride() const { return npt ? (size_t)(nb + 2) * (nb + 2) : (size_t)nb + 2; }
    __device__ size_t cell(int b) const
    {
        return npt ? (size_t)(b / nb + 1) * (nb + 2) + (b % nb + 1) : (size_t)b + 1;
    }
};

// sum over each row of 16 lanes and over the wave, in every lane
__device__ __forceinline__ double mh_row_sum(double v) { return ptmc::group_sum<16>(v); }
__device__ __forceinline__ double mh_wave_sum(double v)
{
    v = mh_row_sum(v);
    v = v + __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// total of one histogram over the workgroup's threads (red: a double per
// wave), complete in thread 0
__device__ double mh_total(const double *H, const MHBins &bins, int n_bins, double *red)
{
    double s = 0.0;
    for (int b = threadIdx.x; b < n_bins; b += MH_THREADS) s = s + H[bins.cell(b)];
    s = mh_wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    for (int w = 1; w < MH_THREADS / 64; ++w) s = s + red[w];
    return s;
}

// histogram totals n_i: one workgroup per (run, temperature)
__global__ void __launch_bounds__(MH_THREADS) mh_total_kernel(MHArgs a)
{
    __shared__ double red[MH_THREADS / 64];
    const MHBins bins(a, blockIdx.x / a.n_temps);
    const double s = mh_total(a.hist + (size_t)blockIdx.x * bins.stride(), bins, a.n_bins, red);
    if (threadIdx.x == 0) a.ncyc[blockIdx.x] = s;
}

// All workgroups of a run have arrived `epoch` times.  The launch is
// cooperative (every workgroup is resident), and a wait that lasts for
// seconds gives up with the error flag, so every wave ends.  Each wave waits
// for its own block sums before the workgroup's barrier: that barrier waits for
// LDS only, and the arrival's release for the stores of its own wave.  The sums
// are agent-scope stores, written past the L2, so the wait is all they need (a
// release fence in every wave would write the L2 back four times, 2.3 us an
// iteration on 79 workgroups).
__device__ bool mh_barrier(const MHArgs &a, int run, unsigned epoch, int *s_ok)
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(&a.count[run], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned want = epoch * (unsigned)a.n_wg;
        int ok = 0;
        for (unsigned n = 0; n < MH_SPIN; ++n) {
            if (__hip_atomic_load(&a.count[run], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want) {
                ok = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (!ok) *a.error = 1;
        *s_ok = ok;
    }
    __syncthreads();
    return *s_ok != 0;
}

// The fixed point of every run.  KEEP: a workgroup keeps its bins' slice of K
// and their terms in LDS; an iteration reads K twice, lanes over bins both
// times (no bank conflicts), and ends in one sum per temperature.  Otherwise
// (slices beyond LDS, and the entry point without workspace) an entry of K is
// formed where it is read, with the same bits.  One workgroup per run where
// the bins are few (NVT: 100-200) or there is no workspace; else the run's
// bins are cut over n_wg workgroups, which exchange their sums once per
// iteration (written and read past the per-XCD L2 by agent-scope accesses,
// two buffers in turn so that one barrier suffices) and each form the same
// free energies.  Sums are formed per block of MH_BINS bins and the blocks
// added in one order, so that results do not depend on the cut.
//
// Bound by the latency of an iteration's chain (two reductions, one exp and
// log per temperature, the barrier), not by arithmetic (VALU issued in 17 % of
// the cycles): 4 us an iteration for 16 runs of 32 x 100 bins, which have no
// barrier (917 -> 162 us a call's kernel against one exponential per temperature
// and bin twice an iteration), 8 us for one run
// of 48 x 10^4 bins on 79 workgroups (98 -> 1.02 ms; 17 us an iteration with
// shuffles instead of row permutations and the exchange's loads one by one).
template <bool KEEP>
__global__ void __launch_bounds__(MH_THREADS) mh_iterate_kernel(MHArgs a)
{
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ int s_ok, s_stop, s_rebase;
    __shared__ double red[MH_THREADS / 64];
    const int R = a.n_temps, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int run = blockIdx.x / a.n_wg, wg = blockIdx.x % a.n_wg;
    const int b0 = wg * a.wg_blk * MH_BINS, nc = min(a.wg_blk * MH_BINS, a.n_bins - b0);
    const int nblk = (nc + MH_BINS - 1) / MH_BINS;
    // blocks are added in q interleaved sequences, then the sequences
    const int q = R < MH_THREADS ? MH_THREADS / R : 1;
    double *fe = reinterpret_cast<double *>(lds);  // R free energies
    double *f0 = fe + R;                           // R those of K
    double *wgt = f0 + R;                          // R: n_i exp(-(f_i - f0_i)), until the bins' ratios are formed
    double *nfe = wgt;                             // R sums, then new free energies, after that
    double *dpart = wgt + R;                       // halves of the bins' sums; the q sequences (R <= MH_THREADS)
    double *end = fe + mh_lds(R, KEEP, false);
    double *ncyc = a.ncyc ? a.ncyc + (size_t)run * R : end;  // end: the entry point without workspace, never KEEP
    const size_t g0 = (size_t)run * a.n_bins + b0;
    double *hs = KEEP ? end : a.hsum + g0;         // nc histogram sums
    double *off = KEEP ? hs + nc : a.off + g0;
    double *ratio = KEEP ? off + nc : a.ratio + g0;  // H_m / D_m
    double *K = ratio + nc;                        // KEEP: R x nc
    const MHBins bins(a, run);
    const double *beta = a.beta + (size_t)run * R;
    const double *H = a.hist + (size_t)run * R * bins.stride();

    for (int i = tid; i < R; i += MH_THREADS) fe[i] = 0.0;
    if (!a.ncyc) {
        for (int i = 0; i < R; ++i) {
            const double s = mh_total(H + (size_t)i * bins.stride(), bins, a.n_bins, red);
            if (tid == 0) ncyc[i] = s;
            __syncthreads();
        }
    }
    auto hist_sum = [&](int m) {
        const double *h = H + bins.cell(b0 + m);
        double s = 0.0;
        for (int i = 0; i < R; ++i) s = s + h[(size_t)i * bins.stride()];
        return s;
    };
    for (int m = tid; m < nc; m += MH_THREADS) hs[m] = hist_sum(m);  // read by the same thread
    if (tid == 0) s_rebase = 1;
    __syncthreads();

    auto term = [&](int i, double h, double o) { return exp(-beta[i] * h - f0[i] - o); };
    // offsets of the current free energies, K from them
    auto rebase = [&]() {
        for (int i = tid; i < R; i += MH_THREADS) f0[i] = fe[i];
        for (int m = tid; m < nc; m += MH_THREADS) {
            const double h = bins.h(b0 + m);
            double o = -1.0e6;
            for (int i = 0; i < R; ++i) o = fmax(o, -beta[i] * h - fe[i]);
            off[m] = o + log(1000.0);
        }
        __syncthreads();
        if constexpr (KEEP)
            for (int e = tid; e < R * nc; e += MH_THREADS) {
                const int i = e / nc, m = e % nc;
                K[e] = term(i, bins.h(b0 + m), off[m]);
            }
    };
    // H_m / D_m: D_m from four interleaved sums over the temperatures, by one
    // thread per bin, or by two where that leaves none idle
    auto ratios = [&]() {
        for (int i = tid; i < R; i += MH_THREADS) wgt[i] = ncyc[i] * exp(f0[i] - fe[i]);
        __syncthreads();
        if constexpr (KEEP) {
            auto pair = [&](int m, int p) {
                double d = 0.0, d1 = 0.0;
                int i = p;
#pragma unroll 4
                for (; i + 2 < R; i += 4) {
                    d = __builtin_fma(wgt[i], K[(size_t)i * nc + m], d);
                    d1 = __builtin_fma(wgt[i + 2], K[(size_t)(i + 2) * nc + m], d1);
                }
                if (i < R) d = __builtin_fma(wgt[i], K[(size_t)i * nc + m], d);
                return d + d1;
            };
            if (nc <= MH_THREADS / 2) {
                const int m = tid % nc, p = tid / nc;
                if (p < 2) dpart[tid] = pair(m, p);
                __syncthreads();
                if (tid < nc) ratio[tid] = hs[tid] / (dpart[tid] + dpart[nc + tid]);
            } else {
                for (int m = tid; m < nc; m += MH_THREADS) ratio[m] = hs[m] / (pair(m, 0) + pair(m, 1));
            }
        } else {
            for (int m = tid; m < nc; m += MH_THREADS) {
                const double h = bins.h(b0 + m), o = off[m];
                double d[4] = {0.0, 0.0, 0.0, 0.0};
                for (int i = 0; i < R; i += 4)
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (i + k < R) d[k] = __builtin_fma(wgt[i + k], term(i + k, h, o), d[k]);
                ratio[m] = hs[m] / ((d[0] + d[2]) + (d[1] + d[3]));
            }
        }
        __syncthreads();
    };

    int it = 0;
    for (it = 1; it <= a.max_iter; ++it) {
        if (s_rebase) rebase();
        __syncthreads();
        ratios();
        double *part = a.n_wg > 1 ? a.part + ((size_t)run * 2 + (it & 1)) * a.n_blk * R : nullptr;
        // block sums, a row of 16 lanes per temperature (all steps of the row
        // sum are lane permutations of the VALU); without a cut they go
        // straight into the sequences, each temperature's by one row in order
        const int row = tid & 15;
        for (int g = 0; g < nblk; ++g) {
            constexpr int U = MH_BINS / 16;
            double rb[U], hb[U], ob[U];  // the lane's bins, for all its temperatures
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int m = min(g * MH_BINS + 16 * u + row, nc - 1);
                rb[u] = ratio[m];
                hb[u] = KEEP ? 0.0 : bins.h(b0 + m);
                ob[u] = KEEP ? 0.0 : off[m];
            }
            for (int i0 = 0; i0 < R; i0 += MH_THREADS / 16) {
                const int i = i0 + tid / 16;
                double s = 0.0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int m = g * MH_BINS + 16 * u + row;
                    if (i < R && m < nc) {
                        double k;
                        if constexpr (KEEP) k = K[(size_t)i * nc + m];
                        else k = term(i, hb[u], ob[u]);
                        s = __builtin_fma(rb[u], k, s);
                    }
                }
                s = mh_row_sum(s);
                if (row == 0 && i < R) {
                    if (a.n_wg > 1) {
                        __hip_atomic_store(&part[(size_t)(wg * a.wg_blk + g) * R + i], s, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    } else {
                        double *acc = q > 1 ? &dpart[(g % q) * R + i] : &nfe[i];
                        *acc = g < q ? 0.0 + s : *acc + s;
                    }
                }
            }
        }
        if (a.n_wg == 1)
            for (int e = nblk * R + tid; e < q * R; e += MH_THREADS) dpart[e] = 0.0;
        if (a.n_wg > 1) {
            if (!mh_barrier(a, run, (unsigned)it, &s_ok)) break;
            for (int e = tid; e < q * R; e += MH_THREADS) {
                const int i = e % R;
                double s = 0.0;
                // 16 loads in flight: each takes about a microsecond
                for (int g = e / R; g < a.n_blk; g += 16 * q) {
                    double v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u)
                        if (g + u * q < a.n_blk)
                            v[u] = __hip_atomic_load(&part[(size_t)(g + u * q) * R + i], __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int u = 0; u < 16; ++u)
                        if (g + u * q < a.n_blk) s = s + v[u];
                }
                if (q > 1) dpart[e] = s;
                else nfe[e] = s;
            }
        }
        __syncthreads();
        for (int i = tid; i < R; i += MH_THREADS) {
            double s = nfe[i];
            if (q > 1) {
                s = dpart[i];
                for (int k = 1; k < q; ++k) s = s + dpart[k * R + i];
            }
            nfe[i] = f0[i] + log(s);
        }
        __syncthreads();
        if (wave == 0) {
            double delta = 0.0, far = 0.0;
            bool nan = false;
            for (int i = lane; i < R; i += 64) {
                const double d = fabs(nfe[i] - fe[i]), r = fabs(nfe[i] - f0[i]);
                delta = delta + d * d;
                far = fmax(far, r);
                nan = nan || !(r == r);
                fe[i] = nfe[i];
            }
            delta = mh_wave_sum(delta);
            const bool move = __ballot(nan || far > MH_REBASE) != 0ull;
            if (lane == 0) {
                s_stop = delta < a.conv;
                s_rebase = move;
            }
        }
        __syncthreads();
        if (s_stop) break;
    }
    if (it > a.max_iter) it = a.max_iter;
    // offsets and ratios of the last free energies, for the output grid
    __syncthreads();
    rebase();
    __syncthreads();
    ratios();
    if constexpr (KEEP) {
        for (int m = tid; m < nc; m += MH_THREADS) {
            a.off[g0 + m] = off[m];
            a.ratio[g0 + m] = ratio[m];
        }
    }
    if (wg == 0) {
        if (a.free_energy)
            for (int i = tid; i < R; i += MH_THREADS) a.free_energy[(size_t)run * R + i] = fe[i];
        if (tid == 0 && a.iterations) a.iterations[run] = it;
    }
}

// Reweighting: one workgroup of T threads per (run, output temperature), one
// pass over the bins.  h is taken from the middle of its range, so that the
// variance loses fewer digits than <h^2> - <h>^2 of the raw values.
template <int T>
__global__ void __launch_bounds__(T) mh_result_kernel(MHArgs a)
{
    __shared__ double red[5][T / 64];
    const int run = blockIdx.x / a.n_res, tid = threadIdx.x;
    const MHBins bins(a, run);
    const double *off = a.off + (size_t)run * a.n_bins, *ratio = a.ratio + (size_t)run * a.n_bins;
    const double bt = a.beta_res[blockIdx.x];
    const double mid = bins.h(a.npt ? (a.n_bin / 2) * a.n_bin + a.n_bin / 2 : a.n_bin / 2);
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};  // 1, E, V, h, h^2
    for (int b = tid; b < a.n_bins; b += T) {
        const double h = bins.h(b);
        const double q = ratio[b] * exp(-bt * h - off[b]);
        const double hc = h - mid;
        s[0] = s[0] + q;
        if (a.npt) {
            s[1] = __builtin_fma(q, bins.energy(b), s[1]);
            s[2] = __builtin_fma(q, bins.volume(b), s[2]);
        }
        s[3] = __builtin_fma(q, hc, s[3]);
        s[4] = __builtin_fma(q, hc * hc, s[4]);
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        s[k] = mh_wave_sum(s[k]);
        if ((tid & 63) == 0) red[k][tid >> 6] = s[k];
    }
    __syncthreads();
    if (tid != 0) return;
    for (int w = 1; w < T / 64; ++w)
        for (int k = 0; k < 5; ++k) s[k] = s[k] + red[k][w];
    const double h1 = s[3] / s[0], h2 = s[4] / s[0], t = a.t_res[blockIdx.x];
    a.c[blockIdx.x] = (h2 - h1 * h1) / (a.k_boltzmann * (t * t));
    if (a.moments) {
        double *mo = a.moments + (size_t)blockIdx.x * 3;
        mo[0] = s[1] / s[0];
        mo[1] = s[2] / s[0];
        mo[2] = h1 + mid;
    }
}

// Device-resident scratch of the allocation-free entry point: the per-bin
// terms of every run of one call (3 n_bin^2 doubles per run: histogram sums,
// offsets and ratios), one copy per GPU for the life of the process.  Every element a call reads it has written first, so nothing needs
// clearing between calls; calls that overlap on one GPU share
// it and race.
static __device__ __align__(256) double npt_scratch[PTMC_NOALLOC_NPT_SCRATCH_DOUBLES];

// device address of npt_scratch on each GPU, looked up once per device
constexpr int MAX_DEVICES = 64;
std::mutex npt_scratch_mutex;
double *npt_scratch_ptr[MAX_DEVICES] = {};

// One device allocation of a call, cut into 256-byte aligned pieces.
struct Arena {
    char *p = nullptr;
    size_t used = 0;
    ~Arena()
    {
        if (p) (void)hipFree(p);
    }
    size_t take(size_t bytes)
    {
        const size_t at = used;
        used += (bytes + 255) & ~(size_t)255;
        return at;
    }
};

struct MHCall {
    int n_runs, n_temps, n_bin, n_res, max_iter, npt;
    const double *beta, *hist, *en_min, *en_max, *v_min, *v_max, *pressure, *beta_res, *t_res;
    double k_boltzmann, conv;
    double *c, *moments, *free_energy;
    int *iterations;
};

#define MHCHK(x)                                     \
    do {                                             \
        if ((x) != hipSuccess) return PTMC_E_DEVICE; \
    } while (0)

// the output grid; a wave per temperature where a run has a few hundred bins
hipError_t mh_results(const MHArgs &a, unsigned n, hipStream_t s)
{
    if (a.n_bins <= 512) hipLaunchKernelGGL(mh_result_kernel<64>, dim3(n), dim3(64), 0, s, a);
    else hipLaunchKernelGGL(mh_result_kernel<256>, dim3(n), dim3(256), 0, s, a);
    return hipGetLastError();
}

int mh_run(const MHCall &q, int device, size_t max_lds)
{
    const size_t R = q.n_temps, B = q.npt ? (size_t)q.n_bin * q.n_bin : (size_t)q.n_bin;
    const size_t cells = q.npt ? (size_t)(q.n_bin + 2) * (q.n_bin + 2) : (size_t)q.n_bin + 2;
    const size_t nR = (size_t)q.n_runs * R, nX = (size_t)q.n_runs * q.n_res;
    int cus = 0;
    MHCHK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    MHArgs a{};
    hipFuncAttributes fa{};  // LDS beside what is asked for
    MHCHK(hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(&mh_iterate_kernel<true>)));
    const MhCut cut = mh_cut(q.n_temps, B, q.n_runs, cus, max_lds - std::min(max_lds, fa.sharedSizeBytes));
    a.n_blk = cut.n_blk;
    a.wg_blk = cut.wg_blk;
    a.n_wg = cut.n_wg;
    const size_t lds = cut.lds;
    const void *fn = cut.keep ? reinterpret_cast<const void *>(&mh_iterate_kernel<true>)
                              : reinterpret_cast<const void *>(&mh_iterate_kernel<false>);
    MHCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // runs of one launch: all, or as many as are resident together when a run has several workgroups
    const int batch = a.n_wg == 1 ? q.n_runs : std::max(1, std::min(q.n_runs, cus / a.n_wg));

    Arena m;
    const size_t o_small = m.take((2 * nX + nR + 5 * (size_t)q.n_runs) * 8);
    const size_t o_hist = m.take(nR * cells * 8);
    const size_t o_out = m.take(((q.moments ? 4 : 1) * nX + nR) * 8 + (size_t)q.n_runs * sizeof(int));
    const size_t o_ncyc = m.take(nR * 8), o_off = m.take((size_t)q.n_runs * B * 8);
    const size_t o_ratio = m.take((size_t)q.n_runs * B * 8);
    const size_t o_hsum = m.take(cut.keep ? 8 : (size_t)q.n_runs * B * 8);
    const size_t o_part = m.take(a.n_wg > 1 ? 2 * nR * a.n_blk * 8 : 8);
    const size_t o_count = m.take(((size_t)q.n_runs + 1) * sizeof(unsigned));
    MHCHK(hipMalloc((void **)&m.p, m.used));

    // the small inputs in one copy
    std::vector<double> in(2 * nX + nR + 5 * (size_t)q.n_runs, 0.0);
    double *w = in.data();
    auto put = [&](const double *from, size_t n) {
        if (from) std::memcpy(w, from, n * 8);
        w += n;
    };
    put(q.beta, nR);
    put(q.beta_res, nX);
    put(q.t_res, nX);
    for (const double *p : {q.en_min, q.en_max, q.v_min, q.v_max, q.pressure}) put(p, q.n_runs);
    MHCHK(hipMemcpyAsync(m.p + o_small, in.data(), in.size() * 8, hipMemcpyHostToDevice, 0));
    MHCHK(hipMemcpyAsync(m.p + o_hist, q.hist, nR * cells * 8, hipMemcpyHostToDevice, 0));
    MHCHK(hipMemsetAsync(m.p + o_count, 0, ((size_t)q.n_runs + 1) * sizeof(unsigned), 0));

    a.n_temps = q.n_temps;
    a.n_bin = q.n_bin;
    a.n_bins = (int)B;
    a.n_res = q.n_res;
    a.max_iter = q.max_iter;
    a.npt = q.npt;
    a.conv = q.conv;
    a.k_boltzmann = q.k_boltzmann;
    double *d = reinterpret_cast<double *>(m.p + o_small);
    a.beta = d;
    a.beta_res = d + nR;
    a.t_res = d + nR + nX;
    a.en_min = d + nR + 2 * nX;
    a.en_max = a.en_min + q.n_runs;
    a.v_min = a.en_max + q.n_runs;
    a.v_max = a.v_min + q.n_runs;
    a.pressure = a.v_max + q.n_runs;
    a.hist = reinterpret_cast<double *>(m.p + o_hist);
    a.c = reinterpret_cast<double *>(m.p + o_out);
    a.moments = q.moments ? a.c + nX : nullptr;
    a.free_energy = a.c + (q.moments ? 4 : 1) * nX;
    a.iterations = reinterpret_cast<int *>(a.free_energy + nR);
    a.ncyc = reinterpret_cast<double *>(m.p + o_ncyc);
    a.off = reinterpret_cast<double *>(m.p + o_off);
    a.ratio = reinterpret_cast<double *>(m.p + o_ratio);
    a.hsum = reinterpret_cast<double *>(m.p + o_hsum);
    a.part = reinterpret_cast<double *>(m.p + o_part);
    a.count = reinterpret_cast<unsigned *>(m.p + o_count);
    a.error = reinterpret_cast<int *>(a.count + q.n_runs);

    hipLaunchKernelGGL(mh_total_kernel, dim3((unsigned)nR), dim3(MH_THREADS), 0, 0, a);
    MHCHK(hipGetLastError());
    for (int r0 = 0; r0 < q.n_runs; r0 += batch) {
        const int nr = std::min(batch, q.n_runs - r0);
        MHArgs b = a;  // the batch's runs
        b.beta += (size_t)r0 * R;
        b.hist += (size_t)r0 * R * cells;
        b.en_min += r0;
        b.en_max += r0;
        b.v_min += r0;
        b.v_max += r0;
        b.pressure += r0;
        b.free_energy += (size_t)r0 * R;
        b.iterations += r0;
        b.ncyc += (size_t)r0 * R;
        b.off += (size_t)r0 * B;
        b.ratio += (size_t)r0 * B;
        if (!cut.keep) b.hsum += (size_t)r0 * B;
        b.part += 2 * (size_t)r0 * a.n_blk * R;
        b.count += r0;
        void *args[] = {&b};
        if (a.n_wg > 1)
            MHCHK(hipLaunchCooperativeKernel(fn, dim3(nr * a.n_wg), dim3(MH_THREADS), args, (unsigned)lds, 0));
        else
            MHCHK(hipLaunchKernel(fn, dim3(nr), dim3(MH_THREADS), args, lds, 0));
    }
    MHCHK(mh_results(a, (unsigned)nX, 0));

    // all results in one copy
    std::vector<char> out(((q.moments ? 4 : 1) * nX + nR) * 8 + (size_t)q.n_runs * sizeof(int));
    int error = 0;
    MHCHK(hipMemcpyAsync(out.data(), m.p + o_out, out.size(), hipMemcpyDeviceToHost, 0));
    if (a.n_wg > 1) MHCHK(hipMemcpyAsync(&error, a.error, sizeof(int), hipMemcpyDeviceToHost, 0));
    MHCHK(hipDeviceSynchronize());
    if (error) return PTMC_E_DEVICE;
    const char *r = out.data();
    auto get = [&](void *to, size_t bytes) {
        if (to) std::memcpy(to, r, bytes);
        r += bytes;
    };
    get(q.c, nX * 8);
    if (q.moments) get(q.moments, 3 * nX * 8);
    get(q.free_energy, nR * 8);
    get(q.iterations, (size_t)q.n_runs * sizeof(int));
    return PTMC_OK;
}

// device and LDS checks of a call; lds: what the description needs at least
int mh_device(int device, size_t lds, size_t &max_lds)
{
    int ndev = 0, v = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PTMC_E_NO_DEVICE;
    if (device < 0 || device >= ndev || hipSetDevice(device) != hipSuccess) return PTMC_E_ARG;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
        return PTMC_E_DEVICE;
    max_lds = (size_t)v;
    return lds > max_lds ? PTMC_E_UNSUPPORTED : PTMC_OK;
}

}  // namespace

extern "C" int ptmc_multihistogram_nvt(int32_t n_runs, int32_t n_temps, int32_t n_bin, const double *beta,
                                       const double *hist, const double *en_min, const double *en_max,
                                       int32_t n_result, const double *beta_result, const double *t_result,
                                       double k_boltzmann, double conv_threshold, int32_t max_iter, double *cv,
                                       double *free_energy, int32_t *iterations, int32_t device)
{
    if (n_runs <= 0 || n_temps <= 0 || n_bin <= 0 || n_result <= 0 || max_iter <= 0 || !beta || !hist ||
        !en_min || !en_max || !beta_result || !t_result || !cv)
        return PTMC_E_ARG;
    size_t max_lds = 0;
    const int rc = mh_device(device, sizeof(double) * (4 * (size_t)n_temps + 3 * (size_t)n_bin) + sizeof(int), max_lds);
    if (rc) return rc;
    const MHCall q{n_runs, n_temps, n_bin, n_result, max_iter, 0, beta, hist, en_min, en_max, nullptr, nullptr,
                   nullptr, beta_result, t_result, k_boltzmann, conv_threshold, cv, nullptr, free_energy, iterations};
    return mh_run(q, device, max_lds);
}

extern "C" int ptmc_multihistogram_npt(int32_t n_runs, int32_t n_temps, int32_t n_bin, const double *beta,
                                       const double *hist, const double *en_min, const double *en_max,
                                       const double *v_min, const double *v_max, const double *pressure,
                                       int32_t n_result, const double *beta_result, const double *t_result,
                                       double k_boltzmann, double conv_threshold, int32_t max_iter, double *cp,
                                       double *moments, double *free_energy, int32_t *iterations, int32_t device)
{
    if (n_runs <= 0 || n_temps <= 0 || n_bin <= 0 || n_result <= 0 || max_iter <= 0 || !beta || !hist ||
        !en_min || !en_max || !v_min || !v_max || !pressure || !beta_result || !t_result || !cp)
        return PTMC_E_ARG;
    if ((int64_t)n_bin * n_bin > (int64_t)1 << 26) return PTMC_E_UNSUPPORTED;
    size_t max_lds = 0;
    const int rc = mh_device(device, sizeof(double) * (4 * (size_t)n_temps + 4) + sizeof(int), max_lds);
    if (rc) return rc;
    const MHCall q{n_runs, n_temps, n_bin, n_result, max_iter, 1, beta, hist, en_min, en_max, v_min, v_max, pressure,
                   beta_result, t_result, k_boltzmann, conv_threshold, cp, moments, free_energy, iterations};
    return mh_run(q, device, max_lds);
}

#undef MHCHK

extern "C" int ptmc_multihistogram_npt_noalloc(int32_t n_runs, int32_t n_temps, int32_t n_bin, const double *beta,
                                               const double *hist, const double *en_min, const double *en_max,
                                               const double *v_min, const double *v_max, const double *pressure,
                                               int32_t n_result, const double *beta_result, const double *t_result,
                                               double k_boltzmann, double conv_threshold, int32_t max_iter,
                                               double *cp, double *moments, double *free_energy,
                                               int32_t *iterations, int32_t device, void *stream)
{
    if (n_runs <= 0 || n_temps <= 0 || n_bin <= 0 || n_result <= 0 || max_iter <= 0 || !beta || !hist ||
        !en_min || !en_max || !v_min || !v_max || !pressure || !beta_result || !t_result || !cp)
        return PTMC_E_ARG;
    if ((int64_t)n_runs * 3 * n_bin * n_bin > (int64_t)PTMC_NOALLOC_NPT_SCRATCH_DOUBLES) return PTMC_E_UNSUPPORTED;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PTMC_E_NO_DEVICE;
    if (device < 0 || device >= ndev || device >= MAX_DEVICES || hipSetDevice(device) != hipSuccess)
        return PTMC_E_ARG;
    int max_lds = 0;
    if (hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
        return PTMC_E_DEVICE;
    if (sizeof(double) * (4 * (size_t)n_temps + 4) + sizeof(int) > (size_t)max_lds) return PTMC_E_UNSUPPORTED;
    const size_t lds = 8 * mh_lds(n_temps, false, true);
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(&mh_iterate_kernel<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return PTMC_E_DEVICE;
    double *scr = nullptr;
    {
        std::lock_guard<std::mutex> lock(npt_scratch_mutex);
        if (!npt_scratch_ptr[device]) {
            void *p = nullptr;
            if (hipGetSymbolAddress(&p, HIP_SYMBOL(npt_scratch)) != hipSuccess || !p) return PTMC_E_DEVICE;
            npt_scratch_ptr[device] = static_cast<double *>(p);
        }
        scr = npt_scratch_ptr[device];
    }
    MHArgs a{};
    a.n_temps = n_temps;
    a.n_bin = n_bin;
    a.n_bins = n_bin * n_bin;
    a.npt = 1;
    a.n_blk = a.wg_blk = (a.n_bins + MH_BINS - 1) / MH_BINS;
    a.n_wg = 1;
    a.n_res = n_result;
    a.max_iter = max_iter;
    a.conv = conv_threshold;
    a.beta = beta;
    a.hist = hist;
    a.en_min = en_min;
    a.en_max = en_max;
    a.v_min = v_min;
    a.v_max = v_max;
    a.pressure = pressure;
    a.beta_res = beta_result;
    a.t_res = t_result;
    a.k_boltzmann = k_boltzmann;
    a.c = cp;
    a.moments = moments;
    a.free_energy = free_energy;
    a.iterations = iterations;
    a.off = scr;
    a.ratio = scr + (size_t)n_runs * a.n_bins;
    a.hsum = scr + 2 * (size_t)n_runs * a.n_bins;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(mh_iterate_kernel<false>, dim3(n_runs), dim3(MH_THREADS), lds, s, a);
    if (hipGetLastError() != hipSuccess) return PTMC_E_DEVICE;
    if (mh_results(a, (unsigned)n_runs * (unsigned)n_result, s) != hipSuccess) return PTMC_E_DEVICE;
    return PTMC_OK;
}
