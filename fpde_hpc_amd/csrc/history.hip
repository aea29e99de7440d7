// History-sum kernels of the Caputo L1 derivative (gfx950).
//
// Storage: D[t][i] = U^{t+1}_i - U^t_i, level-major with node index fastest
// (leading dimension ld, a multiple of 64), so one level is a contiguous row
// and every wavefront reads 64 consecutive nodes.  The step-n history term
// is S_n[i] = sum_{t<n} w(n,t) D[t][i] with the Toeplitz weight
// w(n,t) = omega[n-t-1] (plus the two-level correction added by the step
// kernel).  Kernels here:
//   k_hist_plain   : FP64 streaming sum over a t-range, split over t-chunks
//                    (one partial row per chunk), HBM bound, 8 B per term;
//   k_ref_sum      : the reference "Sum" kernel semantics on level arrays
//                    (fpde_hpc_1d.cpp:1247-1284) behind the OpenCL_* facade;
//   k_gemm_f64     : time-block GEMM  P[ks][r][i] = sum_t omega[n0+r-t-1] D[t][i]
//                    for the B future steps r of a block, on v_mfma_f64_16x16x4;
//   k_pack_split / k_gemm_split : the same GEMM on split bf16/fp16 operands
//                    (hi+lo or hi+mid+lo) with fp32 MFMA accumulation flushed
//                    to fp64 after every 32-level group.
#include "fpde_internal.h"
#include <algorithm>

namespace fpde {

// ---------------------------------------------------------------------------
// Plain FP64 streaming kernel: one workgroup per 512 nodes and t-chunk
// (plain_stream).
__global__ __launch_bounds__(256) void k_hist_plain(const double* __restrict__ D, int64_t ld,
                                                    int nodes, int n, int t_hi, int chunk,
                                                    const double* __restrict__ omega,
                                                    double* __restrict__ part) {
    __shared__ double wwin[kPlainWin];
    plain_stream<256, 4>(D, ld, nodes, n, t_hi, chunk, omega, part, blockIdx.x, blockIdx.y, wwin);
}

// ---------------------------------------------------------------------------
// The whole sum of a short history in one launch: S[i] = sum_t omega[n-t-1]
// D[t][i], a workgroup's 16 waves each taking a sixteenth of the levels of the
// same 128 nodes, the waves' sums added through LDS in level order.  Bound by
// latency: one launch instead of the stream's and the sum of its parts, and a
// wave's levels in flight together, 8 at a time, the first beside the weights.
// Whole calls: 64 levels x 1000 nodes 15.9 -> 14.3 us, 256 x 1000 16.6 -> 15.7,
// 256 x 20000 20.4 -> 18.2; 512 levels 17.0 against 17.9 us (N = 1000), so longer
// histories keep the split over more workgroups, and so do longer lines, where
// the sum is bandwidth again and 16 waves with a few levels each are overhead:
// 65536 nodes x 16 and 256 levels 16.0 and 32.4 against 15.8 and 33.8 us, 10^5
// x 16 and 256 19.1 and 43.7 against 15.8 and 47.2, 10^6 x 1 and 16 48 and 70
// against 21 and 36, 10^7 x 4 432 against 110.
constexpr int kShortLevels = 256, kShortNodes = 65536, kShortWaves = 16;
static bool short_sum(int nodes, int n) { return n <= kShortLevels && nodes <= kShortNodes; }
__global__ __launch_bounds__(64 * kShortWaves) void k_hist_short(double* __restrict__ S, const double* __restrict__ D,
                                                                 int64_t ld, int nodes, int n, int t_hi,
                                                                 const double* __restrict__ omega) {
    __shared__ double w[kShortLevels];                     // w[t] = omega[n-t-1]
    __shared__ double sums[kShortWaves][128];
    constexpr int W = 8;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i2 = (blockIdx.x * 64 + lane) * 2;
    const double* const col = D + (i2 < nodes ? i2 : 0);   // (threads past the nodes still stage weights)
    const int c = (t_hi + kShortWaves - 1) / kShortWaves;
    const int t0 = min(wave * c, t_hi), t1 = min(t0 + c, t_hi);
    double2 d[W];
    auto load = [&](int t) {
#pragma unroll
        for (int j = 0; j < W; j++) {
            d[j] = {0.0, 0.0};
            if (t + j < t1) d[j] = *reinterpret_cast<const double2*>(col + (int64_t)(t + j) * ld);
        }
    };
    load(t0);
    for (int q = tid; q < t_hi; q += 64 * kShortWaves) w[q] = omega[n - q - 1];
    __syncthreads();
    double a0 = 0.0, a1 = 0.0;
    for (int t = t0; t < t1; t += W) {
        double2 e[W];
#pragma unroll
        for (int j = 0; j < W; j++) e[j] = d[j];
        load(t + W);
#pragma unroll
        for (int j = 0; j < W; j++) {
            const double x = t + j < t1 ? w[t + j] : 0.0;
            a0 = fma(x, e[j].x, a0);
            a1 = fma(x, e[j].y, a1);
        }
    }
    sums[wave][2 * lane] = a0;
    sums[wave][2 * lane + 1] = a1;
    __syncthreads();
    const int i = blockIdx.x * 128 + tid;
    if (tid >= 128 || i >= nodes) return;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kShortWaves; k++) s += sums[k][tid];
    S[i] = s;
}

// ---------------------------------------------------------------------------
// The reference Sum kernel, sum_alg 0/1 (fpde_hpc_1d.cpp:1247-1284): newest
// interval first, in chunks of BS levels; sum_alg 1 stops after the first full
// chunk whose weights are all below sum_param in magnitude (the test is on the
// weights alone, so every workgroup finds the cut `lo` first and the sum runs
// over [lo, n)).
// HBM bound: each level is read once (16 bytes per thread and load, 8 levels
// in flight), its difference to the next newer one formed in registers, kb/tau
// divided once per workgroup into LDS windows.  The intervals are split over
// the grid's y as the plain stream's levels are: one thread walking the whole
// history of a node leaves 10^4 nodes on 40 workgroups, each with one load
// in flight (4000 levels x 10^4 nodes: 1775 us, 0.18 TB/s; split: 54 + 4 us,
// 5.9 TB/s).
// Partial rows out[ks * out_stride + i], added newest first by k_ref_combine.
constexpr int kRefWin = 1024;
template <int V>
__global__ __launch_bounds__(256) void k_ref_sum(double* __restrict__ out, int64_t out_stride,
                                                 const double* __restrict__ old, int64_t n, int64_t os, int64_t nodes,
                                                 const double* __restrict__ tau, const double* __restrict__ kb,
                                                 int sum_alg, double sum_param, int bs, int64_t chunk) {
    __shared__ double w[kRefWin];                          // w[l - w0] = kb[l] / tau[l]
    __shared__ unsigned long long cut;                     // first chunk (newest first) wholly below sum_param
    const int tid = threadIdx.x;
    int64_t lo = 0;
    if (sum_alg == 1) {
        const int64_t full = n / bs;
        if (tid == 0) cut = (unsigned long long)full;
        __syncthreads();
        for (int64_t m0 = 0; m0 < full; m0 += 256) {
            const int64_t m = m0 + tid;
            bool below = m < full;
            for (int k = 0; k < bs && below; k++) below = fabs(kb[n - 1 - m * bs - k]) < sum_param;
            if (below) atomicMin(&cut, (unsigned long long)m);
            __syncthreads();
            const bool found = cut < (unsigned long long)(m0 + 256);
            __syncthreads();
            if (found) break;
        }
        if (cut < (unsigned long long)full) lo = n - ((int64_t)cut + 1) * bs;
    }
    const int64_t t0 = max(lo, (int64_t)blockIdx.y * chunk), t1 = min(n, ((int64_t)blockIdx.y + 1) * chunk);
    const int64_t i = ((int64_t)blockIdx.x * 256 + tid) * V;
    const bool ok = i < nodes;                             // the other threads still stage weights
    double acc[V], prev[V];
    auto level = [&](int64_t l, double (&v)[V]) {
        if constexpr (V == 2) {
            const double2 d = *reinterpret_cast<const double2*>(old + l * os + i);
            v[0] = d.x;
            v[1] = d.y;
        } else {
            v[0] = old[l * os + i];
        }
    };
#pragma unroll
    for (int k = 0; k < V; k++) acc[k] = prev[k] = 0.0;
    if (ok && t1 > t0) level(t1, prev);
    for (int64_t w1 = t1; w1 > t0; w1 -= kRefWin) {
        const int64_t w0 = max(t0, w1 - kRefWin);
        __syncthreads();
        for (int q = tid; q < (int)(w1 - w0); q += 256) w[q] = kb[w0 + q] / tau[w0 + q];
        __syncthreads();
        if (!ok) continue;
        int64_t l = w1 - 1;
        for (; l - 7 >= w0; l -= 8) {
            double v[8][V];
#pragma unroll
            for (int j = 0; j < 8; j++) level(l - j, v[j]);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const double wj = w[l - j - w0];
#pragma unroll
                for (int k = 0; k < V; k++) {
                    acc[k] = fma(wj, prev[k] - v[j][k], acc[k]);
                    prev[k] = v[j][k];
                }
            }
        }
        for (; l >= w0; l--) {
            double v[V];
            level(l, v);
#pragma unroll
            for (int k = 0; k < V; k++) {
                acc[k] = fma(w[l - w0], prev[k] - v[k], acc[k]);
                prev[k] = v[k];
            }
        }
    }
    if (!ok) return;
#pragma unroll
    for (int k = 0; k < V; k++)
        if (i + k < nodes) out[(int64_t)blockIdx.y * out_stride + i + k] = acc[k];
}

// S[i] = the parts' sums, newest part first.
__global__ __launch_bounds__(256) void k_ref_combine(double* __restrict__ S, const double* __restrict__ part,
                                                     int splits, int64_t nodes) {
    constexpr int W = 16;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nodes) return;
    double s = 0.0;
    for (int k0 = splits - 1; k0 >= 0; k0 -= W) {
        double v[W];
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = k0 >= j ? part[(int64_t)(k0 - j) * nodes + i] : 0.0;
#pragma unroll
        for (int j = 0; j < W; j++) s += v[j];
    }
    S[i] = s;
}

// ---------------------------------------------------------------------------
// The reference Sum kernel, sum_alg 2 (fpde_hpc_1d.cpp:1285-1302): per node,
// the moments Htmp[id*P + j] += gt^{j+1} coef[j] (old[1][id] - old[0][id])
// (non-finite factors read as 0, as the reference kernel does), then
// S = sum_j v1_j Htmp[id*P + j] / tau[tstep] with the coefficients of
// _kb_row2_fixed_coefs (:1159-1180): v1_0 = gtj^-alpha,
// v1_j = v1_{j-1} (alpha+j-1)/(j gtj).
__global__ __launch_bounds__(256) void k_ref_series(double* __restrict__ S, const double* __restrict__ old,
                                                    int64_t old_size, int64_t os, int64_t nodes,
                                                    const double* __restrict__ tau, int tstep,
                                                    double* __restrict__ Htmp, const double* __restrict__ coef,
                                                    int P, double gtj, double gt, double alpha) {
    int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= nodes) return;
    double ts = 0.0;
    if (old_size >= 2) {
        double cur = old[os + id] - old[id];
        double* h = Htmp + id * P;
        double m = gt;
        for (int j = 0; j < P; j++) {
            double cc = coef[j];
            if (!isfinite(cc)) cc = 0.0;
            double mm = isfinite(m) ? m : 0.0;
            h[j] += mm * cc * cur;
            m *= gt;
        }
        double v1 = pow(gtj, -alpha);
        for (int j = 0; j < P; j++) {
            ts += (isfinite(v1) ? v1 : 0.0) * h[j];
            double i = (double)(j + 1);
            v1 *= -(-alpha - i + 1.0) / (i * gtj);
        }
        ts /= tau[tstep];
    }
    S[id] = ts;
}

fpde_status launch_ref_series(double* S, const double* old, int64_t old_size, int64_t os, int64_t nodes,
                              const double* tau, int tstep, double* Htmp, const double* coef, int P, double gtj,
                              double gt, double alpha, hipStream_t st) {
    if (nodes <= 0) return FPDE_OK;
    hipLaunchKernelGGL(k_ref_series, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, st, S, old, old_size, os,
                       nodes, tau, tstep, Htmp, coef, P, gtj, gt, alpha);
    return FPDE_OK;
}

// ---------------------------------------------------------------------------
// MFMA operand types
typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));

// The two-level corrections corr[2 (n0+r)] D[0] + corr[2 (n0+r)+1] D[1] of a
// block's rows, added to the partial rows of K split 0 (3D: the step then
// reads neither level; corr null: the step kernel adds them itself).
struct GemmCorr {
    const double* corr;        // at 2 n0
    double d0, d1;
    __device__ GemmCorr(const double* c, const double* D0, int64_t ld, int ks, int64_t node, bool ok)
        : corr(ks == 0 ? c : nullptr), d0(0.0), d1(0.0) {
        if (corr && ok) { d0 = D0[node]; d1 = D0[ld + node]; }
    }
    __device__ double operator()(int r, double acc) const {
        return corr ? fma(corr[2 * r + 1], d1, fma(corr[2 * r], d0, acc)) : acc;
    }
};

// FP64 time-block GEMM.  Grid: x = 64-node tiles, y = K splits (t-chunks).
// Block 256 = 4 waves; wave w owns nodes [16w,16w+16) of the tile and all BR
// rows (BR/16 MFMA tiles).  v_mfma_f64_16x16x4f64 operand layout (checked
// on gfx950): A lane l = A[l%16][l/16], B lane l = B[l/16][l%16], and the
// four results of lane l are D[4v + l/16][l%16], v=0..3 (rows interleaved,
// unlike the f32-output MFMAs where lane l holds rows 4(l/16)+v).
template <int BR>
__device__ __forceinline__ void gemm_f64_body(const double* __restrict__ D, int64_t ld, int nodes, int n0, int tc,
                                              int kchunk, const double* __restrict__ omega, double* __restrict__ P,
                                              const double* __restrict__ corr, const double* __restrict__ D0, int bx,
                                              int ks) {
    constexpr int RT = BR / 16;
    constexpr int SLAB = 1024;                  // t-values per LDS weight window
    __shared__ double win[BR + SLAB];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tlo = ks * kchunk;
    const int thi = min(tc, tlo + kchunk);
    const int node = bx * 64 + wave * 16 + (lane & 15);
    const bool node_ok = node < nodes;
    const int kk = lane >> 4;          // k index within the 4-deep MFMA
    d4_t acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) acc[rt] = (d4_t){0.0, 0.0, 0.0, 0.0};
    for (int s0 = tlo; s0 < thi; s0 += SLAB) {
        const int s1 = min(thi, s0 + SLAB);
        // win[q] = omega[n0 - s1 + q], so omega[n0+r-t-1] = win[r - t - 1 + s1]
        const int W = BR + (s1 - s0) - 1;
        __syncthreads();
        for (int q = threadIdx.x; q < W; q += 256) win[q] = omega[n0 - s1 + q];
        __syncthreads();
        // four 4-deep K steps per iteration; the next iteration's four B
        // loads are in flight while this one's MFMAs run
        double bn[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int tt = s0 + 4 * q + kk;
            bn[q] = (tt < s1 && node_ok) ? D[(int64_t)tt * ld + node] : 0.0;
        }
        for (int t = s0; t < s1; t += 16) {
            double b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) b[q] = bn[q];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int tt = t + 16 + 4 * q + kk;
                bn[q] = (tt < s1 && node_ok) ? D[(int64_t)tt * ld + node] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                int tt = t + 4 * q + kk;
                bool ok = tt < s1;
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                    int r = rt * 16 + (lane & 15);
                    double a = ok ? win[r - tt - 1 + s1] : 0.0;
                    acc[rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[q], acc[rt], 0, 0, 0);
                }
            }
        }
    }
    const GemmCorr add(corr, D0, ld, ks, node, node_ok);
    if (node_ok) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                int r = rt * 16 + 4 * v + (lane >> 4);
                P[((int64_t)ks * BR + r) * ld + node] = add(r, acc[rt][v]);
            }
        }
    }
}
template <int BR>
__global__ __launch_bounds__(256) void k_gemm_f64(const double* __restrict__ D, int64_t ld, int nodes, int n0, int tc,
                                                  int kchunk, const double* __restrict__ omega,
                                                  double* __restrict__ P, const double* __restrict__ corr,
                                                  const double* __restrict__ D0) {
    gemm_f64_body<BR>(D, ld, nodes, n0, tc, kchunk, omega, P, corr, D0, blockIdx.x, blockIdx.y);
}

// Several solves' GEMMs of one K split in one launch (y: the solve): the newest
// levels of a batch's solves stand between two step launches, where a launch
// each cost 14 us (8 us and a gap), or 45 us on the hardware queue that shares
// its pipe with the cooperative launches'; six of N = 10^4 in one: 17 us (33).
template <int BR>
__global__ __launch_bounds__(256) void k_gemm_f64_jobs(GemmF64Jobs b) {
    const GemmF64Job& j = b.job[blockIdx.y];
    if ((int)blockIdx.x * 64 >= j.nodes) return;
    gemm_f64_body<BR>(j.D, j.ld, j.nodes, j.n0, j.tc, j.tc, j.omega, j.P, nullptr, nullptr, blockIdx.x, 0);
}

// FP64 time-block GEMM with dense weights (a prescribed non-uniform grid,
// where the weights are not Toeplitz): P[ks][r][i] = sum_t W[r][t] D[t][i],
// W row-major with leading dimension ldw.  Same tiling and MFMA layout as
// k_gemm_f64; the A operand comes from an LDS tile of BR x 64 weights.
template <int BR>
__global__ __launch_bounds__(256) void k_gemm_f64_dense(const double* __restrict__ D, int64_t ld, int nodes,
                                                        int tc, int kchunk, const double* __restrict__ W,
                                                        int64_t ldw, double* __restrict__ P,
                                                    const double* __restrict__ corr, const double* __restrict__ D0) {
    constexpr int RT = BR / 16;
    constexpr int SL = 64;
    __shared__ double win[BR][SL + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ks = blockIdx.y;
    const int tlo = ks * kchunk;
    const int thi = min(tc, tlo + kchunk);
    const int node = blockIdx.x * 64 + wave * 16 + (lane & 15);
    const bool node_ok = node < nodes;
    const int kk = lane >> 4;
    d4_t acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) acc[rt] = (d4_t){0.0, 0.0, 0.0, 0.0};
    for (int s0 = tlo; s0 < thi; s0 += SL) {
        const int s1 = min(thi, s0 + SL);
        __syncthreads();
        for (int q = threadIdx.x; q < BR * SL; q += 256) {
            int r = q / SL, c = q % SL;
            win[r][c] = (s0 + c < s1) ? W[(int64_t)r * ldw + s0 + c] : 0.0;
        }
        __syncthreads();
        for (int t = s0; t < s1; t += 16) {
            double b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                int tt = t + 4 * q + kk;
                b[q] = (tt < s1 && node_ok) ? D[(int64_t)tt * ld + node] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                int tt = t + 4 * q + kk;
                bool ok = tt < s1;
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                    int r = rt * 16 + (lane & 15);
                    double a = ok ? win[r][tt - s0] : 0.0;
                    acc[rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[q], acc[rt], 0, 0, 0);
                }
            }
        }
    }
    const GemmCorr add(corr, D0, ld, ks, node, node_ok);
    if (node_ok) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                int r = rt * 16 + 4 * v + (lane >> 4);
                P[((int64_t)ks * BR + r) * ld + node] = add(r, acc[rt][v]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Split storage.  Group g holds levels [32g, 32g+32); for node i the 32
// values of each component are contiguous: comp[(g*ld + i)*32 + e].  That is
// exactly the B operand of v_mfma_f32_16x16x32_{bf16,f16}: lane l needs
// B[8(l/16)+e][l%16], e=0..7, i.e. 16 contiguous bytes.
// fp16 groups carry a power-of-two scale per (group,node): value = scale*(hi+lo).
template <typename T> struct SplitTraits;
template <> struct SplitTraits<__bf16> {
    typedef bf8_t vec;
    static constexpr bool scaled = false;
};
template <> struct SplitTraits<_Float16> {
    typedef h8_t vec;
    static constexpr bool scaled = true;
};

// Pack levels of complete groups [g_lo, g_hi) from the FP64 history.
// One thread per (group, node).
template <typename T, int NS>
__global__ __launch_bounds__(256) void k_pack_split(const double* __restrict__ D, int64_t ld, int nodes,
                                                    int g_lo, int g_hi, T* __restrict__ c0,
                                                    T* __restrict__ c1, T* __restrict__ c2,
                                                    float* __restrict__ scale) {
    int node = blockIdx.x * 256 + threadIdx.x;
    int g = g_lo + blockIdx.y;
    if (node >= ld || g >= g_hi) return;
    double v[kGroup];
    double mx = 0.0;
#pragma unroll
    for (int e = 0; e < kGroup; e++) {
        v[e] = (node < nodes) ? D[(int64_t)(g * kGroup + e) * ld + node] : 0.0;
        mx = fmax(mx, fabs(v[e]));
    }
    double sc = 1.0;
    if (SplitTraits<T>::scaled) {
        // scaled magnitudes in [2^14, 2^15): hi and lo stay normal fp16 for
        // entries within 2^-10 of the group maximum
        if (mx > 0.0) sc = ldexp(1.0, ilogb(mx) - 14);
        scale[(int64_t)g * ld + node] = (float)sc;
    }
    double inv = 1.0 / sc;
    int64_t base = ((int64_t)g * ld + node) * kGroup;
#pragma unroll
    for (int e = 0; e < kGroup; e++) {
        double x = v[e] * inv;
        T h = (T)(float)x;
        double r = x - (double)(float)h;
        T m = (T)(float)r;
        c0[base + e] = h;
        c1[base + e] = m;
        if (NS == 3) {
            double r2 = r - (double)(float)m;
            c2[base + e] = (T)(float)r2;
        }
    }
}

// A fragments of the split GEMM for the groups [0, tc/32) of one block: the
// weights of rows r < BR against the levels of a group (Toeplitz
// omega[n0+r-t-1], or with DENSE the rows W[r][t] of a prescribed grid),
// split hi/lo(/lo2) into the MFMA A-operand layout (lane l of fragment rt:
// row 16 rt + l%16, levels 8(l/16)..8(l/16)+7 of the group).  They depend on
// the block only, not on the node tile or the K split, so they are formed
// once here instead of in every GEMM workgroup.  Layout: afrag[((g NS + c)
// RT + rt) 64 + lane], ainv[g RT + rt] = 1 / the fragment's power-of-two
// scale (fp16; 1 for bf16).  Grid: one workgroup per group; each wave builds
// whole fragments, so the dense form's fragment maximum is a wave maximum.
template <typename T, int NS, int BR, bool DENSE>
__global__ __launch_bounds__(256) void k_afrag_split(int n0, const double* __restrict__ omega,
                                                     const double* __restrict__ W, int64_t ldw,
                                                     typename SplitTraits<T>::vec* __restrict__ afrag,
                                                     double* __restrict__ ainv) {
    typedef typename SplitTraits<T>::vec vec_t;
    constexpr int RT = BR / 16;
    const int g = blockIdx.x;
    for (int f = threadIdx.x; f < RT * 64; f += 256) {
        const int fl = f & 63, frt = f >> 6;
        const int r = frt * 16 + (fl & 15);
        const int tbase = g * kGroup + 8 * (fl >> 4);
        double wd[8];
#pragma unroll
        for (int e = 0; e < 8; e++) wd[e] = DENSE ? W[(int64_t)r * ldw + tbase + e] : omega[n0 + r - (tbase + e) - 1];
        // fp16: power-of-two scale per fragment so that its largest weight
        // sits in [2^14, 2^15) and the lo parts stay normal.  Toeplitz
        // weights decrease with the lag n0+r-t, so the extremes are at the
        // corners; dense rows take the maximum over the fragment.
        double sa = 1.0;
        if constexpr (SplitTraits<T>::scaled && DENSE) {
            double mx = 0.0;
#pragma unroll
            for (int e = 0; e < 8; e++) mx = fmax(mx, fabs(wd[e]));
            mx = wave_max(mx);
            if (mx > 0.0) sa = ldexp(1.0, 14 - ilogb(mx));
        } else if (SplitTraits<T>::scaled) {
            const int lag_lo = n0 + frt * 16 - (g * kGroup + kGroup - 1);
            const int lag_hi = n0 + frt * 16 + 15 - g * kGroup;
            const double wmax = fmax(fabs(omega[lag_lo - 1]), fabs(omega[lag_hi - 1]));
            if (wmax > 0.0) sa = ldexp(1.0, 14 - ilogb(wmax));
        }
        if (fl == 0) ainv[g * RT + frt] = 1.0 / sa;
        vec_t h, m, l;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const double wv = wd[e] * sa;
            T hh = (T)(float)wv;
            double rr = wv - (double)(float)hh;
            T mm = (T)(float)rr;
            h[e] = hh;
            m[e] = mm;
            if (NS == 3) l[e] = (T)(float)(rr - (double)(float)mm);
        }
        const size_t base = ((size_t)g * NS * RT + frt) * 64 + fl;
        afrag[base] = h;
        afrag[base + RT * 64] = m;
        if (NS == 3) afrag[base + 2 * RT * 64] = l;
    }
}

// The products of one 32-level group, components a (weights) and b (history),
// hi first: one fp32 chain, hi*hi, then the smaller cross products (their
// rounding is 2^-24 of the group sum).
template <typename T, int NS>
__device__ __forceinline__ f4_t split_products(const typename SplitTraits<T>::vec (&a)[NS],
                                               const typename SplitTraits<T>::vec (&b)[NS]) {
    f4_t p = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](int i, int j) {
        if constexpr (SplitTraits<T>::scaled) p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], p, 0, 0, 0);
        else p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], p, 0, 0, 0);
    };
    add(0, 0);
    add(0, 1);
    add(1, 0);
    if constexpr (NS == 3) {
        add(0, 2);
        add(1, 1);
        add(2, 0);
    }
    return p;
}

// Split GEMM.  Grid: x = 64-node tiles, y = K splits.  Per 32-level group:
// wave w (nodes 16w..16w+15) loads its B fragments (one 16-B load per
// component), the A fragments (k_afrag_split) come from LDS, where the block
// stages them for 4 groups at a time, and the products are accumulated in
// fp32 by magnitude class, then flushed to fp64.
template <typename T, int NS, int BR>
__global__ __launch_bounds__(256) void k_gemm_split(const T* __restrict__ c0, const T* __restrict__ c1,
                                                    const T* __restrict__ c2,
                                                    const float* __restrict__ scale, int64_t ld,
                                                    int nodes, int tc, int kchunk,
                                                    const typename SplitTraits<T>::vec* __restrict__ afrag_g,
                                                    const double* __restrict__ ainv_g,
                                                    double* __restrict__ P,
                                                    const double* __restrict__ corr, const double* __restrict__ D0) {
    typedef typename SplitTraits<T>::vec vec_t;
    constexpr int RT = BR / 16;
    constexpr int GB = 4;                                  // groups per LDS batch
    // afrag[comp][gb][rt][lane] : 8 elements each
    __shared__ vec_t afrag[NS][GB][RT][64];
    __shared__ double ainv[GB][RT];                        // 1 / weight scale of a fragment
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ks = blockIdx.y;
    const int glo = (ks * kchunk) / kGroup;
    const int ghi = min(tc, ks * kchunk + kchunk) / kGroup;
    const int node = blockIdx.x * 64 + wave * 16 + (lane & 15);
    const bool node_ok = node < nodes;
    d4_t acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) acc[rt] = (d4_t){0.0, 0.0, 0.0, 0.0};

    // software pipeline: the next batch's B fragments (history) and A
    // fragments (weights) load into registers while this batch computes
    constexpr int AE = GB * RT * 64 / 256;                // A entries per thread per batch
    vec_t bn[GB][NS], an[AE][NS];
    double sn[GB], ain[AE];
    auto load_batch = [&](int gb0) {
#pragma unroll
        for (int gi = 0; gi < GB; gi++) {
            const int g = min(gb0 + gi, ghi - 1);
            const int64_t off = ((int64_t)g * ld + (node_ok ? node : 0)) * kGroup + 8 * (lane >> 4);
            bn[gi][0] = *reinterpret_cast<const vec_t*>(c0 + off);
            bn[gi][1] = *reinterpret_cast<const vec_t*>(c1 + off);
            if (NS == 3) bn[gi][NS - 1] = *reinterpret_cast<const vec_t*>(c2 + off);
            sn[gi] = 1.0;
            if (SplitTraits<T>::scaled) sn[gi] = node_ok ? (double)scale[(int64_t)g * ld + node] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < AE; k++) {
            const int f = threadIdx.x + 256 * k;
            const int fl = f & 63, frt = (f >> 6) % RT, fgb = f / (64 * RT);
            const int g = min(gb0 + fgb, ghi - 1);          // groups past ghi are never used
            const size_t base = ((size_t)g * NS * RT + frt) * 64 + fl;
            an[k][0] = afrag_g[base];
            an[k][1] = afrag_g[base + RT * 64];
            if (NS == 3) an[k][NS - 1] = afrag_g[base + 2 * RT * 64];
            ain[k] = ainv_g[g * RT + frt];
        }
    };
    if (glo < ghi) load_batch(glo);
    for (int gb0 = glo; gb0 < ghi; gb0 += GB) {
        vec_t bfr[GB][NS];
        double bsc[GB];
#pragma unroll
        for (int gi = 0; gi < GB; gi++) {
#pragma unroll
            for (int c = 0; c < NS; c++) bfr[gi][c] = bn[gi][c];
            bsc[gi] = sn[gi];
        }
        __syncthreads();                       // the previous batch is done with the LDS fragments
#pragma unroll
        for (int k = 0; k < AE; k++) {
            const int f = threadIdx.x + 256 * k;
            const int fl = f & 63, frt = (f >> 6) % RT, fgb = f / (64 * RT);
#pragma unroll
            for (int c = 0; c < NS; c++) afrag[c][fgb][frt][fl] = an[k][c];
            if (fl == 0) ainv[fgb][frt] = ain[k];
        }
        if (gb0 + GB < ghi) load_batch(gb0 + GB);
        __syncthreads();
#pragma unroll
        for (int gi = 0; gi < GB; gi++) {
            int g = gb0 + gi;
            if (g >= ghi) break;
            vec_t b[NS];
#pragma unroll
            for (int c = 0; c < NS; c++) b[c] = bfr[gi][c];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                vec_t a[NS];
#pragma unroll
                for (int c = 0; c < NS; c++) a[c] = afrag[c][gi][rt][lane];
                const f4_t p = split_products<T, NS>(a, b);
                double scr = SplitTraits<T>::scaled ? bsc[gi] * ainv[gi][rt] : 1.0;
#pragma unroll
                for (int v = 0; v < 4; v++) acc[rt][v] = fma(scr, (double)p[v], acc[rt][v]);
            }
        }
    }
    const GemmCorr add(corr, D0, ld, ks, node, node_ok);
    if (node_ok) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                int r = rt * 16 + 4 * (lane >> 4) + v;
                P[((int64_t)ks * BR + r) * ld + node] = add(r, acc[rt][v]);
            }
        }
    }
}

// The split GEMM straight from the FP64 history, for one block of steps (the
// direct call): the levels are split into their 16-bit components in the
// registers of the wave that multiplies them, in the values and the order of
// k_pack_split and k_gemm_split, so the results are theirs bit for bit.  One
// pass over 8 B per level and node instead of packing them (8 read, 4 or 6
// written) and reading the components back; where a history serves many
// blocks, as in a solve, packing once is the cheaper way.  HBM bound: a lane's
// 8 levels x 4 groups are in flight while the previous 4 groups' are split and
// multiplied (levels 8 (l/16) + e of the group at node l%16 are just its B
// operand, so nothing goes through LDS but the weights' fragments).
// 9984 levels x 10^4 nodes, B = 64, bf16: 182-201 us (4.2 TB/s) and 13 us for the
// sum of 13 splits, against 259 us packing, 105 us GEMM, 64 sums of 3.5 us and
// about 17 ms of allocating and freeing the components; whole call 19.1 -> 0.20 ms.
template <typename T, int NS, int BR>
__global__ __launch_bounds__(256) void k_gemm_split_direct(const double* __restrict__ D, int64_t ld, int nodes, int tc,
                                                           int kchunk,
                                                           const typename SplitTraits<T>::vec* __restrict__ afrag_g,
                                                           const double* __restrict__ ainv_g,
                                                           double* __restrict__ P) {
    typedef typename SplitTraits<T>::vec vec_t;
    constexpr int RT = BR / 16;
    constexpr int GB = 2;                                  // groups per batch
    __shared__ vec_t afrag[NS][GB][RT][64];
    __shared__ double ainv[GB][RT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ks = blockIdx.y;
    const int glo = (ks * kchunk) / kGroup;
    const int ghi = min(tc, ks * kchunk + kchunk) / kGroup;
    const int node = blockIdx.x * 64 + wave * 16 + (lane & 15);
    const bool node_ok = node < nodes;
    const double* col = D + (node_ok ? node : 0) + (int64_t)(8 * (lane >> 4)) * ld;
    d4_t acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) acc[rt] = (d4_t){0.0, 0.0, 0.0, 0.0};
    constexpr int AE = (GB * RT * 64 + 255) / 256;         // A entries per thread per batch
    double dn[GB][8];
    vec_t an[AE][NS];
    double ain[AE];
    auto load_batch = [&](int gb0) {
#pragma unroll
        for (int gi = 0; gi < GB; gi++) {
            const double* d = col + (int64_t)min(gb0 + gi, ghi - 1) * kGroup * ld;
#pragma unroll
            for (int e = 0; e < 8; e++) dn[gi][e] = d[(int64_t)e * ld];
        }
#pragma unroll
        for (int k = 0; k < AE; k++) {
            const int f = min((int)threadIdx.x + 256 * k, GB * RT * 64 - 1);
            const int fl = f & 63, frt = (f >> 6) % RT, fgb = f / (64 * RT);
            const int g = min(gb0 + fgb, ghi - 1);          // groups past ghi are never used
            const size_t base = ((size_t)g * NS * RT + frt) * 64 + fl;
            an[k][0] = afrag_g[base];
            an[k][1] = afrag_g[base + RT * 64];
            if (NS == 3) an[k][NS - 1] = afrag_g[base + 2 * RT * 64];
            ain[k] = ainv_g[g * RT + frt];
        }
    };
    if (glo < ghi) load_batch(glo);
    for (int gb0 = glo; gb0 < ghi; gb0 += GB) {
        double dv[GB][8];
#pragma unroll
        for (int gi = 0; gi < GB; gi++)
#pragma unroll
            for (int e = 0; e < 8; e++) dv[gi][e] = node_ok ? dn[gi][e] : 0.0;
        __syncthreads();                       // the previous batch is done with the LDS fragments
#pragma unroll
        for (int k = 0; k < AE; k++) {
            const int f = threadIdx.x + 256 * k;
            const int fl = f & 63, frt = (f >> 6) % RT, fgb = f / (64 * RT);
            if (f < GB * RT * 64) {
#pragma unroll
                for (int c = 0; c < NS; c++) afrag[c][fgb][frt][fl] = an[k][c];
                if (fl == 0) ainv[fgb][frt] = ain[k];
            }
        }
        if (gb0 + GB < ghi) load_batch(gb0 + GB);
        __syncthreads();
#pragma unroll
        for (int gi = 0; gi < GB; gi++) {
            if (gb0 + gi >= ghi) break;
            // this lane's levels in components (k_pack_split)
            double sc = 1.0;
            if constexpr (SplitTraits<T>::scaled) {
                double mx = 0.0;
#pragma unroll
                for (int e = 0; e < 8; e++) mx = fmax(mx, fabs(dv[gi][e]));
                mx = fmax(mx, __shfl_xor(mx, 16));          // the group's other 24 levels of the node
                mx = fmax(mx, __shfl_xor(mx, 32));
                if (mx > 0.0) sc = ldexp(1.0, ilogb(mx) - 14);
            }
            const double inv = 1.0 / sc;
            vec_t b[NS];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const double x = dv[gi][e] * inv;
                const T h = (T)(float)x;
                const double r = x - (double)(float)h;
                const T m = (T)(float)r;
                b[0][e] = h;
                b[1][e] = m;
                if (NS == 3) b[NS - 1][e] = (T)(float)(r - (double)(float)m);
            }
            const double bsc = SplitTraits<T>::scaled ? (node_ok ? (double)(float)sc : 0.0) : 1.0;
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                vec_t a[NS];
#pragma unroll
                for (int c = 0; c < NS; c++) a[c] = afrag[c][gi][rt][lane];
                const f4_t p = split_products<T, NS>(a, b);
                const double scr = SplitTraits<T>::scaled ? bsc * ainv[gi][rt] : 1.0;
#pragma unroll
                for (int v = 0; v < 4; v++) acc[rt][v] = fma(scr, (double)p[v], acc[rt][v]);
            }
        }
    }
    if (node_ok) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                int r = rt * 16 + 4 * (lane >> 4) + v;
                P[((int64_t)ks * BR + r) * ld + node] = acc[rt][v];
            }
        }
    }
}

// P[r][i] = the K splits' partial rows added in split order, for every row of a
// block at once (one row: the parts of a streamed history sum).
__global__ __launch_bounds__(256) void k_part_sum(double* __restrict__ P, const double* __restrict__ part, int splits,
                                                  int rows, int64_t ld, int nodes) {
    constexpr int W = 16;
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int r = blockIdx.y;
    if (i >= nodes) return;
    double s = 0.0;
    for (int k0 = 0; k0 < splits; k0 += W) {
        double v[W];
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = (k0 + j < splits) ? part[((int64_t)(k0 + j) * rows + r) * ld + i] : 0.0;
#pragma unroll
        for (int j = 0; j < W; j++) s += v[j];
    }
    P[(int64_t)r * ld + i] = s;
}

fpde_status launch_part_sum(double* P, const double* part, int splits, int rows, int64_t ld, int nodes,
                            hipStream_t st) {
    hipLaunchKernelGGL(k_part_sum, dim3((unsigned)((nodes + 255) / 256), (unsigned)rows), dim3(256), 0, st, P, part,
                       splits, rows, ld, nodes);
    FPDE_HIP_TRY(hipGetLastError());
    return FPDE_OK;
}

// ---------------------------------------------------------------------------
// Fold the K-split partial rows of a GEMM block into split 0, in place and in
// split order: P[0][r][i] = ((P[0] + P[1]) + P[2]) + ..., so a 1D step reads
// one far value per node.  The splits of one (r, i) load as one batch of
// independent loads.  (Folding inside the GEMM by its last-arriving
// workgroup per tile needs an agent-scope release per workgroup, an L2
// write-back on gfx950, and measured slower than this pass.)
__global__ __launch_bounds__(256) void k_part_reduce(double* __restrict__ P, int splits, int rows,
                                                     int64_t ld, int nodes) {
    constexpr int W = 16;
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int r = blockIdx.y;
    if (i >= nodes || r >= rows) return;
    double s = P[(int64_t)r * ld + i];
    for (int k0 = 1; k0 < splits; k0 += W) {
        double v[W];
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = (k0 + j < splits) ? P[((int64_t)(k0 + j) * rows + r) * ld + i] : 0.0;
#pragma unroll
        for (int j = 0; j < W; j++)
            if (k0 + j < splits) s += v[j];
    }
    P[(int64_t)r * ld + i] = s;
}

fpde_status launch_part_reduce(double* P, int splits, int rows, int64_t ld, int nodes, hipStream_t st) {
    if (splits <= 1 || nodes <= 0) return FPDE_OK;
    dim3 grid((unsigned)((nodes + 255) / 256), (unsigned)rows);
    hipLaunchKernelGGL(k_part_reduce, grid, dim3(256), 0, st, P, splits, rows, ld, nodes);
    return FPDE_OK;
}

// ---------------------------------------------------------------------------
// Host launchers
// t-split plan of the plain stream: enough workgroups to fill the chip
// (~4096 with the node tiles), each streaming >= 32 levels; at most
// max_splits partial rows.  Returns the number of partial rows.
int hist_plain_plan(int nodes, int t_hi, int* chunk_out, int max_splits) {
    if (t_hi <= 0 || nodes <= 0) { if (chunk_out) *chunk_out = 0; return 0; }
    int tiles = (nodes + 511) / 512;
    int want = (4096 + tiles - 1) / tiles;
    if (want > max_splits) want = max_splits;
    if (want < 1) want = 1;
    int chunk = (t_hi + want - 1) / want;
    if (chunk < 32) chunk = 32;
    if (chunk_out) *chunk_out = chunk;
    return (t_hi + chunk - 1) / chunk;
}

fpde_status launch_hist_plain(const double* D, int64_t ld, int nodes, int n, int t_hi,
                              const double* omega, double* part, int* splits_out,
                              hipStream_t st, int max_splits) {
    int chunk = 0;
    const int splits = hist_plain_plan(nodes, t_hi, &chunk, max_splits);
    *splits_out = splits;
    if (splits == 0) return FPDE_OK;
    int tiles = (nodes + 511) / 512;
    dim3 grid(tiles, splits);
    hipLaunchKernelGGL(k_hist_plain, grid, dim3(256), 0, st, D, ld, nodes, n, t_hi, chunk, omega, part);
    return FPDE_OK;
}

// Partial rows of launch_hist_sum (a short history needs none).
int hist_sum_rows(int nodes, int n) { return short_sum(nodes, n) ? 0 : hist_plain_plan(nodes, n, nullptr); }

fpde_status launch_hist_sum(double* S, const double* D, int64_t ld, int nodes, int n, const double* omega,
                            double* part, hipStream_t st) {
    if (nodes <= 0) return FPDE_OK;
    if (short_sum(nodes, n)) {
        hipLaunchKernelGGL(k_hist_short, dim3((unsigned)((nodes + 127) / 128)), dim3(64 * kShortWaves), 0, st, S, D, ld,
                           nodes, n, n, omega);
        FPDE_HIP_TRY(hipGetLastError());
        return FPDE_OK;
    }
    int splits = 0;
    fpde_status rc = launch_hist_plain(D, ld, nodes, n, n, omega, part, &splits, st);
    if (rc != FPDE_OK) return rc;
    // 16 rows to a memory trip: with the 3D history combine, which takes 8 (16
    // cost it 1 to 3% of a 3D solve), whole calls took 19.6 us at 300 nodes x
    // 2000 levels (19.0 so) and 25.4 at 1000 x 4000 (24.6)
    return launch_part_sum(S, part, splits, 1, ld, nodes, st);
}

// Parts of the reference Sum: about 2048 workgroups with the 512-node tiles
// (8 per CU; 512 to 4096 measured alike), each walking at least 64 intervals:
// whole calls of 4000 x 10^4 took 71, 71 and 67 us with at least 16, 32 and 64,
// of 8000 x 300 41, 29 and 24 us (fewer partial rows to add), of 500 x 5000
// 18.5, 18.3 and 19.6 us.
int ref_sum_splits(int64_t nodes, int64_t intervals) {
    if (nodes <= 0) return 1;
    const int64_t tiles = (nodes + 511) / 512;
    int64_t s = std::min<int64_t>((2048 + tiles - 1) / tiles, intervals / 64);
    return (int)std::max<int64_t>(1, std::min<int64_t>(s, kPlainMaxSplits));
}

fpde_status launch_ref_sum(double* S, const double* old, int64_t old_size, int64_t os,
                           int64_t nodes, const double* tau, const double* kb, int sum_alg,
                           double sum_param, int bs, double* part, hipStream_t st) {
    if (nodes <= 0) return FPDE_OK;
    if (bs < 1) bs = 1;
    const int64_t n = old_size >= 2 ? old_size - 1 : 0;
    int splits = ref_sum_splits(nodes, n);
    if (splits > 1 && !part) { set_error("reference sum: no room for the partial rows"); return FPDE_ERR_ARG; }
    const int64_t chunk = std::max<int64_t>((n + splits - 1) / splits, 1);
    splits = (int)std::max<int64_t>((n + chunk - 1) / chunk, 1);
    double* out = splits > 1 ? part : S;
    // two nodes per thread where every level's rows are 16-byte aligned and the
    // last pair stays inside the level
    const bool pairs = os % 2 == 0 && ((uintptr_t)old & 15) == 0;
    const int64_t per = pairs ? 512 : 256;
    const dim3 grid((unsigned)((nodes + per - 1) / per), (unsigned)splits);
    if (pairs)
        hipLaunchKernelGGL(k_ref_sum<2>, grid, dim3(256), 0, st, out, nodes, old, n, os, nodes, tau, kb, sum_alg,
                           sum_param, bs, chunk);
    else
        hipLaunchKernelGGL(k_ref_sum<1>, grid, dim3(256), 0, st, out, nodes, old, n, os, nodes, tau, kb, sum_alg,
                           sum_param, bs, chunk);
    if (splits > 1)
        hipLaunchKernelGGL(k_ref_combine, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, st, S, part, splits,
                           nodes);
    return FPDE_OK;
}

// K splits for a GEMM over t < tc: enough workgroups to cover the chip
// (>= ~2048 with the node tiles), at most 16 partial rows per output.
int gemm_max_splits(int64_t nodes) {
    int64_t tiles = (nodes + 63) / 64;
    int64_t s = (2048 + tiles - 1) / tiles;
    return (int)(s < 1 ? 1 : (s > 16 ? 16 : s));
}

static void gemm_split_plan(int tc, int64_t nodes, int* kchunk, int* splits, int max_splits) {
    int ks = gemm_max_splits(nodes);
    if (max_splits > 0 && ks > max_splits) ks = max_splits;
    int ch = (tc + ks - 1) / ks;
    ch = ((ch + 31) / 32) * 32;
    if (ch < 32) ch = 32;
    *kchunk = ch;
    *splits = (tc + ch - 1) / ch;
}

fpde_status launch_gemm_f64_dense(const double* D, int64_t ld, int nodes, int tc, int block, const double* W,
                                  int64_t ldw, double* P, int* splits_out, hipStream_t st, int max_splits, const double* corr,
                              const double* D0) {
    if (tc <= 0) { *splits_out = 0; return FPDE_OK; }
    int kchunk, splits;
    gemm_split_plan(tc, nodes, &kchunk, &splits, max_splits);
    dim3 grid((unsigned)((nodes + 63) / 64), (unsigned)splits);
    switch (block) {
        case 16: hipLaunchKernelGGL(k_gemm_f64_dense<16>, grid, dim3(256), 0, st, D, ld, nodes, tc, kchunk, W, ldw, P, corr, D0); break;
        case 32: hipLaunchKernelGGL(k_gemm_f64_dense<32>, grid, dim3(256), 0, st, D, ld, nodes, tc, kchunk, W, ldw, P, corr, D0); break;
        case 64: hipLaunchKernelGGL(k_gemm_f64_dense<64>, grid, dim3(256), 0, st, D, ld, nodes, tc, kchunk, W, ldw, P, corr, D0); break;
        case 128: hipLaunchKernelGGL(k_gemm_f64_dense<128>, grid, dim3(256), 0, st, D, ld, nodes, tc, kchunk, W, ldw, P, corr, D0); break;
        default: set_error("block must be 16, 32, 64 or 128"); return FPDE_ERR_ARG;
    }
    *splits_out = splits;
    FPDE_HIP_TRY(hipGetLastError());
    return FPDE_OK;
}

fpde_status launch_gemm_f64(const double* D, int64_t ld, int nodes, int n0, int tc, int block,
                            const double* omega, double* P, int* splits_out, hipStream_t st, int max_splits, const double* corr,
                              const double* D0) {
    if (tc <= 0) { *splits_out = 0; return FPDE_OK; }
    int kchunk, splits;
    gemm_split_plan(tc, nodes, &kchunk, &splits, max_splits);
    dim3 grid((nodes + 63) / 64, splits);
    size_t lds = 0;
    switch (block) {
        case 16: hipLaunchKernelGGL(k_gemm_f64<16>, grid, dim3(256), lds, st, D, ld, nodes, n0, tc, kchunk, omega, P, corr, D0); break;
        case 32: hipLaunchKernelGGL(k_gemm_f64<32>, grid, dim3(256), lds, st, D, ld, nodes, n0, tc, kchunk, omega, P, corr, D0); break;
        case 64: hipLaunchKernelGGL(k_gemm_f64<64>, grid, dim3(256), lds, st, D, ld, nodes, n0, tc, kchunk, omega, P, corr, D0); break;
        case 128: hipLaunchKernelGGL(k_gemm_f64<128>, grid, dim3(256), lds, st, D, ld, nodes, n0, tc, kchunk, omega, P, corr, D0); break;
        default: set_error("block must be 16, 32, 64 or 128"); return FPDE_ERR_ARG;
    }
    *splits_out = splits;
    return FPDE_OK;
}

fpde_status launch_gemm_f64_jobs(const GemmF64Jobs& b, int count, int block, hipStream_t st) {
    int nodes = 0;
    if (count < 1) return FPDE_OK;
    if (count > kMaxBatch) { set_error("GEMM jobs: at most 32"); return FPDE_ERR_ARG; }
    for (int j = 0; j < count; j++) nodes = std::max(nodes, b.job[j].nodes);
    const dim3 grid((unsigned)((nodes + 63) / 64), (unsigned)count);
    switch (block) {
        case 16: hipLaunchKernelGGL(k_gemm_f64_jobs<16>, grid, dim3(256), 0, st, b); break;
        case 32: hipLaunchKernelGGL(k_gemm_f64_jobs<32>, grid, dim3(256), 0, st, b); break;
        case 64: hipLaunchKernelGGL(k_gemm_f64_jobs<64>, grid, dim3(256), 0, st, b); break;
        case 128: hipLaunchKernelGGL(k_gemm_f64_jobs<128>, grid, dim3(256), 0, st, b); break;
        default: set_error("block must be 16, 32, 64 or 128"); return FPDE_ERR_ARG;
    }
    FPDE_HIP_TRY(hipGetLastError());
    return FPDE_OK;
}

template <typename T, int NS>
static fpde_status pack_t(const double* D, int64_t ld, int nodes, int g_lo, int g_hi, void* c0,
                          void* c1, void* c2, float* scale, hipStream_t st) {
    dim3 grid((unsigned)((ld + 255) / 256), g_hi - g_lo);
    hipLaunchKernelGGL((k_pack_split<T, NS>), grid, dim3(256), 0, st, D, ld, nodes, g_lo, g_hi, (T*)c0,
                       (T*)c1, (T*)c2, scale);
    return FPDE_OK;
}

fpde_status launch_pack_split(int mode, const double* D, int64_t ld, int nodes, int g_lo, int g_hi,
                              void* c0, void* c1, void* c2, float* scale, hipStream_t st) {
    if (g_hi <= g_lo) return FPDE_OK;
    switch (mode) {
        case HIST_SPLIT_BF16: return pack_t<__bf16, 2>(D, ld, nodes, g_lo, g_hi, c0, c1, c2, scale, st);
        case HIST_SPLIT_F16: return pack_t<_Float16, 2>(D, ld, nodes, g_lo, g_hi, c0, c1, c2, scale, st);
        case HIST_SPLIT_BF16X3: return pack_t<__bf16, 3>(D, ld, nodes, g_lo, g_hi, c0, c1, c2, scale, st);
        default: set_error("bad split mode"); return FPDE_ERR_ARG;
    }
}

template <typename T, int NS, int BR>
static void gemm_split_t(dim3 grid, hipStream_t st, const void* c0, const void* c1, const void* c2,
                         const float* scale, int64_t ld, int nodes, int n0, int tc, int kchunk,
                         const double* omega, const double* W, int64_t ldw, void* afrag, double* ainv, double* P,
                         const double* corr, const double* D0) {
    typedef typename SplitTraits<T>::vec vec_t;
    if (W)
        hipLaunchKernelGGL((k_afrag_split<T, NS, BR, true>), dim3(tc / kGroup), dim3(256), 0, st, n0, omega, W, ldw,
                           (vec_t*)afrag, ainv);
    else
        hipLaunchKernelGGL((k_afrag_split<T, NS, BR, false>), dim3(tc / kGroup), dim3(256), 0, st, n0, omega, W, ldw,
                           (vec_t*)afrag, ainv);
    hipLaunchKernelGGL((k_gemm_split<T, NS, BR>), grid, dim3(256), 0, st, (const T*)c0, (const T*)c1, (const T*)c2,
                       scale, ld, nodes, tc, kchunk, (const vec_t*)afrag, (const double*)ainv, P, corr, D0);
}

template <typename T, int NS>
static fpde_status gemm_split_b(int block, dim3 grid, hipStream_t st, const void* c0, const void* c1,
                                const void* c2, const float* scale, int64_t ld, int nodes, int n0,
                                int tc, int kchunk, const double* omega, const double* W, int64_t ldw,
                                void* afrag, double* ainv, double* P, const double* corr, const double* D0) {
    switch (block) {
        case 16: gemm_split_t<T, NS, 16>(grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        case 32: gemm_split_t<T, NS, 32>(grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        case 64: gemm_split_t<T, NS, 64>(grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        case 128: gemm_split_t<T, NS, 128>(grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        default: set_error("block must be 16, 32, 64 or 128"); return FPDE_ERR_ARG;
    }
    return FPDE_OK;
}

template <typename T, int NS, int BR>
static void gemm_direct_t(dim3 grid, hipStream_t st, const double* D, int64_t ld, int nodes, int n0, int tc, int kchunk,
                          const double* omega, void* afrag, double* ainv, double* P) {
    typedef typename SplitTraits<T>::vec vec_t;
    hipLaunchKernelGGL((k_afrag_split<T, NS, BR, false>), dim3(tc / kGroup), dim3(256), 0, st, n0, omega, (const double*)nullptr,
                       (int64_t)0, (vec_t*)afrag, ainv);
    hipLaunchKernelGGL((k_gemm_split_direct<T, NS, BR>), grid, dim3(256), 0, st, D, ld, nodes, tc, kchunk,
                       (const vec_t*)afrag, (const double*)ainv, P);
}

template <typename T, int NS>
static fpde_status gemm_direct_b(int block, dim3 grid, hipStream_t st, const double* D, int64_t ld, int nodes, int n0,
                                 int tc, int kchunk, const double* omega, void* afrag, double* ainv, double* P) {
    switch (block) {
        case 16: gemm_direct_t<T, NS, 16>(grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        case 32: gemm_direct_t<T, NS, 32>(grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        case 64: gemm_direct_t<T, NS, 64>(grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        case 128: gemm_direct_t<T, NS, 128>(grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        default: set_error("block must be 16, 32, 64 or 128"); return FPDE_ERR_ARG;
    }
    return FPDE_OK;
}

fpde_status launch_gemm_split_direct(int mode, const double* D, int64_t ld, int nodes, int n0, int tc, int block,
                                     const double* omega, void* afrag, double* ainv, double* P, int* splits_out,
                                     hipStream_t st) {
    if (tc <= 0) { *splits_out = 0; return FPDE_OK; }
    if (tc % kGroup != 0) { set_error("split GEMM needs a group-aligned cut"); return FPDE_ERR_ARG; }
    int kchunk, splits;
    gemm_split_plan(tc, nodes, &kchunk, &splits, 0);
    const dim3 grid((nodes + 63) / 64, splits);
    fpde_status rc;
    switch (mode) {
        case HIST_SPLIT_BF16: rc = gemm_direct_b<__bf16, 2>(block, grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        case HIST_SPLIT_F16: rc = gemm_direct_b<_Float16, 2>(block, grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        case HIST_SPLIT_BF16X3: rc = gemm_direct_b<__bf16, 3>(block, grid, st, D, ld, nodes, n0, tc, kchunk, omega, afrag, ainv, P); break;
        default: set_error("bad split mode"); return FPDE_ERR_ARG;
    }
    *splits_out = splits;
    return rc;
}

size_t split_afrag_bytes(int mode, int block, int groups) {
    const size_t ns = (mode == HIST_SPLIT_BF16X3) ? 3 : 2;
    return (size_t)groups * ns * (size_t)(block / 16) * 64 * 16;
}

fpde_status launch_gemm_split(int mode, const void* c0, const void* c1, const void* c2,
                              const float* scale, int64_t ld, int nodes, int n0, int tc, int block,
                              const double* omega, const double* W, int64_t ldw, void* afrag, double* ainv,
                              double* P, int* splits_out, hipStream_t st, int max_splits, const double* corr,
                              const double* D0) {
    if (tc <= 0) { *splits_out = 0; return FPDE_OK; }
    if (tc % kGroup != 0) { set_error("split GEMM needs a group-aligned cut"); return FPDE_ERR_ARG; }
    if (W && ldw < tc) { set_error("split GEMM: dense weight rows shorter than the cut"); return FPDE_ERR_ARG; }
    if (!afrag || !ainv) { set_error("split GEMM: no fragment workspace"); return FPDE_ERR_ARG; }
    int kchunk, splits;
    gemm_split_plan(tc, nodes, &kchunk, &splits, max_splits);
    dim3 grid((nodes + 63) / 64, splits);
    fpde_status rc;
    switch (mode) {
        case HIST_SPLIT_BF16: rc = gemm_split_b<__bf16, 2>(block, grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        case HIST_SPLIT_F16: rc = gemm_split_b<_Float16, 2>(block, grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        case HIST_SPLIT_BF16X3: rc = gemm_split_b<__bf16, 3>(block, grid, st, c0, c1, c2, scale, ld, nodes, n0, tc, kchunk, omega, W, ldw, afrag, ainv, P, corr, D0); break;
        default: set_error("bad split mode"); return FPDE_ERR_ARG;
    }
    *splits_out = splits;
    return rc;
}

}  // namespace fpde
