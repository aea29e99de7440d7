// 3D locally-one-dimensional step (gfx950), fpde_hpc_1d.cpp:5144-5626.
//
// Field layout idx = z + n*(x + n*y): depth z fastest (the reference's N axis,
// idx() at :1181).  One step = three sweeps in the reference order:
//   y (m3d_c=2, carries the history term), x (m3d_c=1), z (m3d_c=0); with
//   split3d odd each of the three carries a third of it.
// Every sweep solves, line by line, L*(U - U_in) = div_axis(K grad U) + H
// with coefficients evaluated at the field the sweep starts from.
//  - y and x lines: one thread per line (adjacent threads = adjacent z, so
//    every load is coalesced) running the reference Thomas recurrences
//    al1/bt1/U1 (:4002-4027, :4585-4590, :4672-4725) with zero flux at both
//    ends (Al[1]=1, Bt[1]=0; bcN()=0), coefficients precomputed per node;
//  - z lines: one workgroup per line, one node per thread, PCR in LDS,
//    Dirichlet top / zero-flux bottom; it also writes D[n] = U^{n+1}-U^n.
// With the space-fractional scheme every sweep also takes kap and the line
// sums E of its own axis (space.hip, k_space3d).
#include "fpde_internal.h"
#include <algorithm>

namespace fpde {

// K and 1/C of every node at the current field.
__device__ __forceinline__ void coef3d_body(const double* __restrict__ U, int n, double h, double ksat, int mode,
                                            double* __restrict__ K, double* __restrict__ iC, int bid) {
    int64_t id = (int64_t)bid * 256 + threadIdx.x;
    int64_t nn = (int64_t)n * n * n;
    if (id >= nn) return;
    int z = (int)(id % n);
    double k, ic;
    vgm_coefs(U[id], z * h, ksat, mode, k, ic);
    K[id] = k;
    iC[id] = ic;
}
__global__ __launch_bounds__(256) void k_coef3d(const double* __restrict__ U, int n, double h,
                                                double ksat, int mode, double* __restrict__ K,
                                                double* __restrict__ iC) {
    coef3d_body(U, n, h, ksat, mode, K, iC, blockIdx.x);
}

// Lateral sweep, thread per line.  axis 1 = x (stride n), 2 = y (stride n*n).
// Scratch Al/Bt: [n+1][nlines], coalesced.  The row data of a line are
// fetched 16 rows at a time (independent loads) ahead of the recurrence, and
// the back substitution fetches Al/Bt the same way, so a line costs ~n/16
// memory round trips instead of n.
// Space-fractional scheme (E != nullptr): the diffusion part of the rows is
// scaled by kap = Dg kb(gamma,i-1,i,i) and Om carries -inv_dw_dh E (E: the
// line sums of k_space3d), as in the 1D rows.
__global__ __launch_bounds__(256) void k_lateral3d(const double* U, double* Uout, const double* __restrict__ K,
                                                   const double* __restrict__ iC,
                                                   const double* __restrict__ H, int n, int axis,
                                                   double h2inv, double L, double* __restrict__ Al,
                                                   double* __restrict__ Bt, double kap,
                                                   const double* __restrict__ E) {
    constexpr int R = 16;
    int line = blockIdx.x * 256 + threadIdx.x;
    int nlines = n * n;
    if (line >= nlines) return;
    int z = line % n, o = line / n;
    int64_t base, stride;
    if (axis == 2) { base = z + (int64_t)n * o; stride = (int64_t)n * n; }   // (z,x=o), along y
    else { base = z + (int64_t)n * n * o; stride = n; }                        // (z,y=o), along x
    const int N = n - 1;
    // al1 with Al[1]=1 (lateral, :4021), bt1 with Bt[1]=bc0()=0 (:4511)
    double al = 1.0, bt = 0.0;
    Al[(int64_t)1 * nlines + line] = al;
    Bt[(int64_t)1 * nlines + line] = bt;
    double Kprev = K[base];
    for (int i0 = 1; i0 < N; i0 += R) {
        double kk[R], ic[R], uu[R], hh[R], ee[R];
#pragma unroll
        for (int j = 0; j < R; j++) {
            int i = i0 + j;
            bool ok = i < N;
            int64_t id = base + stride * (ok ? i : 0);
            kk[j] = ok ? K[id] : 0.0;
            ic[j] = ok ? iC[id] : 0.0;
            uu[j] = ok ? U[id] : 0.0;
            hh[j] = (ok && H) ? H[id] : 0.0;
            ee[j] = (ok && E) ? E[id] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < R; j++) {
            int i = i0 + j;
            if (i < N) {
                double Km = Kprev, Kp = kk[j];
                double A_ = Km * ic[j] * h2inv * kap;
                double B_ = Kp * ic[j] * h2inv * kap;
                double R_ = ic[j] * ((Kp * h2inv) + (Km * h2inv)) * kap + L;
                double Om = -L * uu[j] + hh[j];
                if (E) Om -= ic[j] * ee[j];
                double aln = B_ / (R_ - A_ * al);
                bt = (aln / B_) * (A_ * bt - Om);
                al = aln;
                Al[(int64_t)(i + 1) * nlines + line] = al;
                Bt[(int64_t)(i + 1) * nlines + line] = bt;
                Kprev = Kp;
            }
        }
    }
    // zero-flux end, U1 :4704-4720 with bcN()=0
    double uN;
    if (fabs(bt) > 1e-15) uN = (fabs(1.0 - al) > 1e-15) ? bt / (1.0 - al) : U[base + stride * (N - 1)];
    else uN = (fabs(1.0 - al) > 1e-15) ? 0.0 : U[base + stride * (N - 1)];
    Uout[base + stride * N] = uN;
    double u = uN;
    for (int i1 = N - 1; i1 >= 0; i1 -= R) {
        double aa[R], bb[R];
#pragma unroll
        for (int j = 0; j < R; j++) {
            int i = i1 - j;
            bool ok = i >= 0;
            aa[j] = ok ? Al[(int64_t)(i + 1) * nlines + line] : 0.0;
            bb[j] = ok ? Bt[(int64_t)(i + 1) * nlines + line] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < R; j++) {
            int i = i1 - j;
            if (i >= 0) {
                u = aa[j] * u + bb[j];
                Uout[base + stride * i] = u;
            }
        }
    }
}


// Depth sweep: block = one z line, one node per thread (blockDim = n rounded
// up to 64, n <= 256).  PCR on rows normalised to b = 1 with ping-pong LDS
// buffers (one barrier and one reciprocal per level).  From V; writes U^{n+1}
// over U^n and the history level D[t] = U^{n+1} - U^n.
__global__ __launch_bounds__(256) void k_zline3d(const double* __restrict__ V, double* __restrict__ U,
                                                 const double* __restrict__ utop, int n, double h,
                                                 double h2inv, double ksat, int mode, double L,
                                                 double* __restrict__ Dlev, double kap,
                                                 const double* __restrict__ E,
                                                 const double* __restrict__ H) {
    __shared__ double a[2][256], c[2][256], d[2][256], sK[256];
    const int tid = threadIdx.x;
    const int line = blockIdx.x;                   // x + n*y
    const int64_t base = (int64_t)n * line;
    const bool act = tid < n;
    double u = 0.0, k = 0.0, ic = 0.0, uprev = 0.0;
    if (act) {
        u = V[base + tid];
        uprev = U[base + tid];
        vgm_coefs(u, tid * h, ksat, mode, k, ic);
        sK[tid] = k;
    }
    double top = utop[line];
    __syncthreads();
    if (act) {
        double ar, br, cr, dr;
        if (tid == 0) { ar = 0.0; br = 1.0; cr = 0.0; dr = top; }
        else if (tid == n - 1) { ar = -1.0; br = 1.0; cr = 0.0; dr = 0.0; }
        else {
            double Km = sK[tid - 1], Kp = k;
            ar = Km * ic * h2inv * kap;
            cr = Kp * ic * h2inv * kap;
            br = -(ic * ((Kp * h2inv) + (Km * h2inv)) * kap + L);
            dr = -L * u + (H ? H[base + tid] : 0.0);
            if (E) dr -= ic * E[base + tid];
        }
        double ib = 1.0 / br;
        a[0][tid] = ar * ib; c[0][tid] = cr * ib; d[0][tid] = dr * ib;
    }
    __syncthreads();
    int p = 0;
    for (int delta = 1; delta < n; delta <<= 1) {
        if (act) {
            double aq = a[p][tid], cq = c[p][tid], dq = d[p][tid];
            double am = 0, cm = 0, dm = 0, ap = 0, cp = 0, dp = 0;
            if (tid - delta >= 0) { am = a[p][tid - delta]; cm = c[p][tid - delta]; dm = d[p][tid - delta]; }
            if (tid + delta < n) { ap = a[p][tid + delta]; cp = c[p][tid + delta]; dp = d[p][tid + delta]; }
            double inv = 1.0 / (1.0 - aq * cm - cq * ap);
            a[1 - p][tid] = -aq * am * inv;
            c[1 - p][tid] = -cq * cp * inv;
            d[1 - p][tid] = (dq - aq * dm - cq * dp) * inv;
        }
        __syncthreads();
        p = 1 - p;
    }
    if (act) {
        double un = d[p][tid];
        int64_t id = base + tid;
        U[id] = un;
        Dlev[id] = un - uprev;
    }
}

// Partitioned sweeps (n <= 128, L > 0): a workgroup takes kLineGroup lines and
// cuts each into segments of kSegRows rows, one thread each (thread = line +
// kLineGroup * segment, so that the lateral axes' loads are coalesced over the
// 16 consecutive z).  The line's system is the reference one (lateral: zero
// flux at both ends, U_0 = U_1: Al_1 = 1, Bt_1 = 0, fpde_hpc_1d.cpp:4021,
// :4511; U_N = U_{N-1}: the bottom of U1, :4704-4720; depth: U_0 = u_top) and
// the rows of A_/B/R/Om between.  The reference's 1e-15 guards on the bottom
// row act on singular lines (|1 - Al_N| <= 1e-15, which L > 0 rules out: every
// row is diagonally dominant) and on a bottom value within 1e-15 of zero,
// where the two differ by less than that absolute amount.
//
// What bounds them: FP64 issue (VGM coefficients and row eliminations, about
// half of the time) and memory, one after the other unless several workgroups
// of a CU are in different phases.  So the rows per thread are few enough for
// 4 waves per SIMD: segments of 8 rows with their last rows reduced cyclically
// over the segments (4 levels, one reciprocal each, through LDS) instead of
// segments of 16 with every thread walking all segments' ends (256 registers,
// 2 waves per SIMD, a reciprocal per segment).  n = 128: lateral sweep 23.0 ->
// 16.4 us, depth sweep 34 -> 21.3 us.
constexpr int kSegRows = 8, kSegMax = 16, kLineGroup = kLinesHost3D;
struct Line3DLds { double v[2][3][kSegMax][kLineGroup]; };

// Solve the lines of a workgroup, rows a x_{i-1} + b x_i + c x_{i+1} = d of
// segment sg (of W; a = 0 on the line's first row, c = 0 on its last) of line l:
// a segment's first rows are eliminated against its last one (two couplings as
// right-hand sides), the last ones reduced cyclically.  Called by all threads;
// L.v[0] is free on entry.
__device__ __forceinline__ void line3d_solve(const double (&a)[kSegRows], const double (&b)[kSegRows],
                                             const double (&c)[kSegRows], const double (&d)[kSegRows], int l, int sg,
                                             int W, Line3DLds& L, double (&x)[kSegRows]) {
#pragma clang fp contract(off)
    constexpr int S = kSegRows;
    double q[S - 1], y[S - 1];                      // q: c' of the elimination, then z
    {
        const double inv = rcp_nr(b[0]);
        q[0] = c[0] * inv;
        x[0] = d[0] * inv;
        y[0] = -a[0] * inv;
    }
#pragma unroll
    for (int j = 1; j < S - 1; j++) {
        const double inv = rcp_nr(fma(-a[j], q[j - 1], b[j]));
        q[j] = c[j] * inv;
        x[j] = fma(-a[j], x[j - 1], d[j]) * inv;
        y[j] = -(a[j] * y[j - 1]) * inv;
    }
    q[S - 2] = -q[S - 2];
#pragma unroll
    for (int j = S - 3; j >= 0; j--) {
        x[j] = fma(-q[j], x[j + 1], x[j]);
        y[j] = fma(-q[j], y[j + 1], y[j]);
        q[j] = -(q[j] * q[j + 1]);
    }
    L.v[0][0][sg][l] = x[0];
    L.v[0][1][sg][l] = y[0];
    L.v[0][2][sg][l] = q[0];
    __syncthreads();
    double xn = 0.0, yn = 0.0, zn = 0.0;
    if (sg + 1 < W) { xn = L.v[0][0][sg + 1][l]; yn = L.v[0][1][sg + 1][l]; zn = L.v[0][2][sg + 1][l]; }
    double A = a[S - 1], C = c[S - 1], D;
    {
        const double inv = rcp_nr(fma(C, yn, fma(A, q[S - 2], b[S - 1])));
        D = fma(-C, xn, fma(-A, x[S - 2], d[S - 1])) * inv;
        A = (A * y[S - 2]) * inv;
        C = (C * zn) * inv;
    }
    int par = 1;
    for (int s = 1; s < W; s <<= 1) {
        L.v[par][0][sg][l] = A;
        L.v[par][1][sg][l] = C;
        L.v[par][2][sg][l] = D;
        __syncthreads();
        double am = 0.0, cm = 0.0, dm = 0.0, ap = 0.0, cp = 0.0, dp = 0.0;
        if (sg >= s) { am = L.v[par][0][sg - s][l]; cm = L.v[par][1][sg - s][l]; dm = L.v[par][2][sg - s][l]; }
        if (sg + s < W) { ap = L.v[par][0][sg + s][l]; cp = L.v[par][1][sg + s][l]; dp = L.v[par][2][sg + s][l]; }
        const double inv = rcp_nr(fma(-C, ap, fma(-A, cm, 1.0)));
        D = fma(-C, dp, fma(-A, dm, D)) * inv;
        A = -(A * am) * inv;
        C = -(C * cp) * inv;
        par ^= 1;
    }
    L.v[par][0][sg][l] = D;
    __syncthreads();
    const double xl = sg > 0 ? L.v[par][0][sg - 1][l] : 0.0;
    x[S - 1] = D;
#pragma unroll
    for (int j = 0; j < S - 1; j++) x[j] = fma(q[j], D, fma(y[j], xl, x[j]));
}

// Rows of a segment from its U, K, 1/C and the right-hand sides' other terms
// rhs = H - E/C (row i = 8 sg + j); rows past the line are x = 0, coupled to
// nothing.  K of the segment to the left comes through LDS.
__device__ __forceinline__ void line3d_rows(const double (&u)[kSegRows], const double (&K)[kSegRows],
                                            const double (&iC)[kSegRows], const double (&rhs)[kSegRows], int n, int l,
                                            int sg, double h2inv, double lam, double kap, bool depth, double top,
                                            Line3DLds& L, double (&a)[kSegRows], double (&b)[kSegRows],
                                            double (&c)[kSegRows], double (&d)[kSegRows]) {
#pragma clang fp contract(off)
    L.v[1][0][sg][l] = K[kSegRows - 1];
    __syncthreads();
    double Km = sg > 0 ? L.v[1][0][sg - 1][l] : 0.0;
#pragma unroll
    for (int j = 0; j < kSegRows; j++) {
        const int i = kSegRows * sg + j;
        const bool inner = i >= 1 && i < n - 1;
        const double g = iC[j] * h2inv * kap;
        a[j] = inner ? Km * g : (i == n - 1 ? -1.0 : 0.0);
        c[j] = inner ? K[j] * g : (i == 0 && !depth ? -1.0 : 0.0);
        b[j] = inner ? -fma(g, K[j] + Km, lam) : 1.0;
        d[j] = inner ? fma(-lam, u[j], rhs[j]) : (i == 0 ? top : 0.0);
        Km = K[j];
    }
}

// Lateral (y or x) sweep from Uin to Uout (the same field or another).
// K, iC: the coefficients at Uin from a coefficient pass, or nullptr: then the
// sweep evaluates them itself (every node of a lateral line has the same depth
// z0 h), the same values the pass would store.
__device__ __forceinline__ void lateral3d_seg_body(const double* Uin, double* Uout, const double* K, const double* iC,
                                                   const double* H, int n, int axis, double h2inv, double lam,
                                                   double kap, const double* E, double h, double ksat, int mode,
                                                   int bid) {
#pragma clang fp contract(off)
    __shared__ Line3DLds L;
    const int tid = threadIdx.x;
    const int l = tid % kLineGroup, sg = tid / kLineGroup;
    const int line = bid * kLineGroup + l;
    const int ln = min(line, n * n - 1);
    const int z0 = ln % n, o = ln / n;
    int64_t base, stride;
    if (axis == 2) { base = z0 + (int64_t)n * o; stride = (int64_t)n * n; }   // (z,x=o), along y
    else { base = z0 + (int64_t)n * n * o; stride = n; }                        // (z,y=o), along x
    const int W = (n + kSegRows - 1) / kSegRows;
    const double zd = z0 * h;
    auto at = [&](int j) { return base + stride * min(kSegRows * sg + j, n - 1); };   // (rows past the line: its last)
    double u[kSegRows], r[kSegRows], k[kSegRows], ic[kSegRows];
#pragma unroll
    for (int j = 0; j < kSegRows; j++) u[j] = Uin[at(j)];
#pragma unroll
    for (int j = 0; j < kSegRows; j++) r[j] = H ? H[at(j)] : 0.0;
#pragma unroll
    for (int j = 0; j < kSegRows; j++) {
        if (K) { k[j] = K[at(j)]; ic[j] = iC[at(j)]; }
        else vgm_coefs(u[j], zd, ksat, mode, k[j], ic[j]);
        if (E) r[j] = fma(-ic[j], E[at(j)], r[j]);
    }
    double a[kSegRows], b[kSegRows], c[kSegRows], d[kSegRows], x[kSegRows];
    line3d_rows(u, k, ic, r, n, l, sg, h2inv, lam, kap, false, 0.0, L, a, b, c, d);
    line3d_solve(a, b, c, d, l, sg, W, L, x);
    if (line >= n * n) return;
#pragma unroll
    for (int j = 0; j < kSegRows; j++)
        if (kSegRows * sg + j < n) Uout[at(j)] = x[j];
}
constexpr int kSegThreads = kSegMax * kLineGroup;
__global__ __launch_bounds__(kSegThreads, 4) void k_lateral3d_seg(const double* Uin, double* Uout, const double* K,
                                                                  const double* iC, const double* H, int n, int axis,
                                                                  double h2inv, double lam, double kap,
                                                                  const double* E, double h, double ksat, int mode) {
    lateral3d_seg_body(Uin, Uout, K, iC, H, n, axis, h2inv, lam, kap, E, h, ksat, mode, blockIdx.x);
}

// Depth (z) sweep from V: the new U over U^n, D[n] = U - U^n.  The lines are
// contiguous, so rows go between memory (coalesced) and the threads' segments
// through LDS.
__device__ __forceinline__ void zline3d_seg_body(const double* V, double* U, const double* utop, int n, double h,
                                                 double h2inv, double ksat, int mode, double lam, double* Dlev,
                                                 double kap, const double* E, const double* Kin, const double* iCin,
                                                 const double* H, int bid) {
#pragma clang fp contract(off)
    constexpr int LD = kSegRows * kSegMax + 1;          // odd row stride: the 16 lines hit distinct banks
    __shared__ Line3DLds L;
    __shared__ double sU[kLineGroup][LD];
    const int tid = threadIdx.x, T = blockDim.x;
    const int l = tid % kLineGroup, sg = tid / kLineGroup;
    const int line0 = bid * kLineGroup;
    const int nl = min(kLineGroup, n * n - line0);        // lines of this group
    const int64_t base0 = (int64_t)n * line0;
    const int W = (n + kSegRows - 1) / kSegRows;
    const int total = nl * n;                             // <= kSegRows T
    // this thread's elements tid + T k of the group's rows, line and row of each
    const int dl = T / n, di = T % n, l_first = tid / n, i_first = tid % n;
    auto elements = [&](auto&& f) {
        int ll = l_first, ii = i_first;
#pragma unroll
        for (int k = 0; k < kSegRows; k++) {
            if (tid + T * k < total) f(k, ll, ii);
            ll += dl;
            ii += di;
            if (ii >= n) { ii -= n; ll++; }
        }
    };
    // a field's values of this thread's rows (rows past the line and lines past
    // the group: of the last one)
    auto stage = [&](const double* src, double (&to)[kSegRows]) {
        double t[kSegRows];
        elements([&](int k, int, int) { t[k] = src[base0 + tid + T * k]; });
        elements([&](int k, int ll, int ii) { sU[ll][ii] = t[k]; });
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kSegRows; j++) to[j] = sU[min(l, nl - 1)][min(kSegRows * sg + j, n - 1)];
    };
    double u[kSegRows], r[kSegRows], k[kSegRows], ic[kSegRows], uold[kSegRows];
    stage(V, u);
    elements([&](int q, int, int) { uold[q] = U[base0 + tid + T * q]; });
    if (Kin) {
        __syncthreads();
        stage(Kin, k);
        __syncthreads();
        stage(iCin, ic);
    } else {
#pragma unroll
        for (int j = 0; j < kSegRows; j++)
            vgm_coefs(u[j], min(kSegRows * sg + j, n - 1) * h, ksat, mode, k[j], ic[j]);
    }
#pragma unroll
    for (int j = 0; j < kSegRows; j++) r[j] = 0.0;
    if (H) {
        __syncthreads();
        stage(H, r);
    }
    if (E) {
        double e[kSegRows];
        __syncthreads();
        stage(E, e);
#pragma unroll
        for (int j = 0; j < kSegRows; j++) r[j] = fma(-ic[j], e[j], r[j]);
    }
    const double top = utop[line0 + min(l, nl - 1)];
    double a[kSegRows], b[kSegRows], c[kSegRows], d[kSegRows], x[kSegRows];
    line3d_rows(u, k, ic, r, n, l, sg, h2inv, lam, kap, true, top, L, a, b, c, d);
    line3d_solve(a, b, c, d, l, sg, W, L, x);
    // (every thread has read its staged rows: line3d_rows and line3d_solve synchronise)
#pragma unroll
    for (int j = 0; j < kSegRows; j++)
        if (l < nl && kSegRows * sg + j < n) sU[l][kSegRows * sg + j] = x[j];
    __syncthreads();
    elements([&](int q, int ll, int ii) {
        const double un = sU[ll][ii];
        U[base0 + tid + T * q] = un;
        Dlev[base0 + tid + T * q] = un - uold[q];
    });
}
__global__ __launch_bounds__(kSegThreads, 4) void k_zline3d_seg(const double* V, double* U, const double* utop, int n,
                                                                double h, double h2inv, double ksat, int mode,
                                                                double lam, double* Dlev, double kap, const double* E,
                                                                const double* Kin, const double* iCin,
                                                                const double* H) {
    zline3d_seg_body(V, U, utop, n, h, h2inv, ksat, mode, lam, Dlev, kap, E, Kin, iCin, H, blockIdx.x);
}


// History term of NV nodes (id: their indexes): the partial rows, the near
// levels, W of them loaded together, the corrections; the same order of sums
// whatever NV and W.
template <int NV, int W>
__device__ __forceinline__ void hist3d_sum(const Hist3D& h, const int64_t (&id)[NV], double (&S)[NV]) {
#pragma clang fp contract(off)
    double far[NV], nr0[NV], nr1[NV];
#pragma unroll
    for (int q = 0; q < NV; q++) far[q] = nr0[q] = nr1[q] = 0.0;
    for (int r0 = 0; r0 < h.rows; r0 += W) {
        double v[W][NV];
#pragma unroll
        for (int j = 0; j < W; j++)
#pragma unroll
            for (int q = 0; q < NV; q++) v[j][q] = r0 + j < h.rows ? h.part[(r0 + j) * h.part_stride + id[q]] : 0.0;
#pragma unroll
        for (int j = 0; j < W; j++)
#pragma unroll
            for (int q = 0; q < NV; q++) far[q] += v[j][q];
    }
    for (int t0 = h.lo; t0 < h.n; t0 += W) {
        double v[W][NV], w[W];
#pragma unroll
        for (int j = 0; j < W; j++) {
            const bool ok = t0 + j < h.n;
#pragma unroll
            for (int q = 0; q < NV; q++) v[j][q] = ok ? h.D[(int64_t)(t0 + j) * h.ld + id[q]] : 0.0;
            w[j] = ok ? h.omega[h.n - t0 - j - 1] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < W; j += 2)
#pragma unroll
            for (int q = 0; q < NV; q++) {
                nr0[q] = fma(w[j], v[j][q], nr0[q]);
                nr1[q] = fma(w[j + 1], v[j + 1][q], nr1[q]);
            }
    }
    const double c0 = h.corr && h.n >= 1 ? h.corr[0] : 0.0, c1 = h.corr && h.n >= 2 ? h.corr[1] : 0.0;
#pragma unroll
    for (int q = 0; q < NV; q++) {
        double cr = 0.0;
        if (h.corr && h.n >= 1) cr = c0 * h.D[id[q]];
        if (h.corr && h.n >= 2) cr = fma(c1, h.D[h.ld + id[q]], cr);
        S[q] = (far[q] + (nr0[q] + nr1[q])) + cr;
    }
}

// S of every node, times hscale (1, or 1/3 when every sweep carries a third of
// the term): HBM bound, one pass over the rows and levels of hist3d_sum.
__device__ __forceinline__ void hist_combine_body(double* __restrict__ S, const Hist3D& h, int64_t nodes,
                                                  double hscale, int bid) {
    const int64_t id[1] = {(int64_t)bid * 256 + threadIdx.x};
    if (id[0] >= nodes) return;
    double s[1];
    hist3d_sum<1, 8>(h, id, s);
    S[id[0]] = s[0] * hscale;
}
__global__ __launch_bounds__(256) void k_hist_combine(double* __restrict__ S, Hist3D h, int64_t nodes, double hscale) {
    hist_combine_body(S, h, nodes, hscale, blockIdx.x);
}

// Near levels folded ahead, at most 32 at a time: every level of the range is
// read once and added to the partial rows of the steps that follow, so a step
// reads one row and at most 7 levels.  HBM bound.  Ranges and targets: when
// c levels of the near field are complete, 2^k the lowest bit of c (2^k >= 8),
// the last 2^k levels go to the next 2^k steps, so that at any step the binary
// digits of c name the ranges its row holds.  Per step of a 64-step block 4.5
// rows and levels move here and 3.5 levels are read directly (16-level groups
// folded for the rest of the block: 4 and 7.5, and a row of their own).  128^3,
// per step: folds 14 us (5.3 TB/s) and history term 17.9 us against 49 us.
// The weights of a batch of targets stand in the lanes of one register (a
// Toeplitz vector) or one per target (the steps' own rows) and are broadcast
// from there: one scalar load per weight and target took 200 cycles each.
__device__ inline double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
template <int LEN, bool TOEPLITZ>
__device__ __forceinline__ void fold3d_levels(const Fold3D& f, int64_t i, bool ok, int lo, bool first) {
#pragma clang fp contract(off)
    constexpr int PB = 8;
    const int lane = threadIdx.x & 63;
    double dv[LEN], row[PB];
#pragma unroll
    for (int k = 0; k < LEN; k++) dv[k] = f.D[(int64_t)(lo + k) * f.ld + i];
    auto load = [&](int p0) {
#pragma unroll
        for (int j = 0; j < PB; j++)
            row[j] = !first && p0 + j < f.p_hi ? f.part[(int64_t)(p0 + j - f.n0) * f.ld + i] : 0.0;
    };
    load(f.p_lo);
    for (int p0 = f.p_lo; p0 < f.p_hi; p0 += PB) {
        double acc[PB], wv[TOEPLITZ ? 1 : PB];
        // weight of level lo + k at step p0 + j: lane LEN - 1 + j - k of wv[0], or lane k of wv[j]
        if constexpr (TOEPLITZ) {
            wv[0] = f.omega[min(p0 - lo - LEN + lane, f.p_hi - lo - 2)];
        } else {
#pragma unroll
            for (int j = 0; j < PB; j++) {
                const int p = min(p0 + j, f.p_hi - 1);
                wv[j] = f.omega[(int64_t)(p - f.n0) * f.omega_stride + p - lo - 1 - min(lane, LEN - 1)];
            }
        }
#pragma unroll
        for (int j = 0; j < PB; j++) acc[j] = row[j];
        if (p0 + PB < f.p_hi) load(p0 + PB);
#pragma unroll
        for (int k = 0; k < LEN; k++)
#pragma unroll
            for (int j = 0; j < PB; j++)
                acc[j] = fma(TOEPLITZ ? lane_value(wv[0], LEN - 1 + j - k) : lane_value(wv[TOEPLITZ ? 0 : j], k), dv[k],
                             acc[j]);
#pragma unroll
        for (int j = 0; j < PB; j++)
            if (ok && p0 + j < f.p_hi) f.part[(int64_t)(p0 + j - f.n0) * f.ld + i] = acc[j];
    }
}
__device__ inline int batch_slot(const int* first, int count, int bid) {
    int j = 0;
    while (j + 1 < count && bid >= first[j + 1]) j++;
    return j;
}
__global__ __launch_bounds__(256) void k_fold3d(Fold3DBatch b) {
    const int j = batch_slot(b.first, b.count, blockIdx.x);
    const Fold3D& f = b.row[j];
    const int64_t i0 = (int64_t)((int)blockIdx.x - b.first[j]) * 256 + threadIdx.x;
    const bool ok = i0 < f.nodes;                      // (idle lanes still hold weights)
    const int64_t i = ok ? i0 : 0;
    auto fold = [&](auto toeplitz) {
        constexpr bool T = decltype(toeplitz)::value;
        if (f.len == 8) fold3d_levels<8, T>(f, i, ok, f.lo, f.first);
        else if (f.len == 16) fold3d_levels<16, T>(f, i, ok, f.lo, f.first);
        else
            for (int q = 0; q < f.len; q += 32) fold3d_levels<32, T>(f, i, ok, f.lo + q, f.first && q == 0);
    };
    if (f.omega_stride == 0) fold(std::true_type{});
    else fold(std::false_type{});
}

// Series-compressed history (sum_alg 2): add the newest interval dnew to the
// moments and sum the series, S[i] = sum_j v_j (H[j][i] += c_j dnew[i]);
// dnew == nullptr (step 0) gives S = 0.
__global__ __launch_bounds__(256) void k_series3d(double* __restrict__ S, double* __restrict__ H, int P,
                                                  const double* __restrict__ dnew,
                                                  const double* __restrict__ ser_c,
                                                  const double* __restrict__ ser_v, int64_t nodes, int64_t ld,
                                                  double hscale) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nodes) return;
    if (!dnew) { S[i] = 0.0; return; }
    S[i] = series_update(H, ld, i, P, dnew[i], ser_c, ser_v) * hscale;
}

// ---------------------------------------------------------------------------
// Batched step of several 3D solves: the same bodies, each workgroup mapped to
// (solve j, its local block) by the prefix counts of the table.
__global__ __launch_bounds__(256) void k_hist_combine_batch(Lod3DBatch b) {
    const int j = batch_slot(b.first_node, b.count, blockIdx.x);
    const Lod3DRow& r = b.row[j];
    hist_combine_body(r.S, r.hist, r.nodes, r.hscale, (int)blockIdx.x - b.first_node[j]);
}

// y sweep (axis 2) carries the history term; the x sweep (axis 1) a third of
// it with split3d odd
__global__ __launch_bounds__(kSegThreads, 4) void k_lateral3d_batch(Lod3DBatch b, int axis) {
    const int j = batch_slot(b.first_line, b.count, blockIdx.x);
    const Lod3DRow& r = b.row[j];
    lateral3d_seg_body(axis == 2 ? r.U : r.V, r.V, r.Kl, r.iCl, (axis == 2 || r.split) ? r.S : nullptr, r.n, axis, r.h2inv, r.L,
                           r.kap, r.E, r.h, r.ksat, r.coef_mode, (int)blockIdx.x - b.first_line[j]);
}

__global__ __launch_bounds__(kSegThreads, 4) void k_zline3d_batch(Lod3DBatch b) {
    const int j = batch_slot(b.first_line, b.count, blockIdx.x);
    const Lod3DRow& r = b.row[j];
    zline3d_seg_body(r.V, r.U, r.utop, r.n, r.h, r.h2inv, r.ksat, r.coef_mode, r.L, r.Dlev, r.kap, r.E,
                     r.Kz, r.iCz, r.split ? r.S : nullptr, (int)blockIdx.x - b.first_line[j]);
}

// threads of a workgroup of the partitioned sweeps (whole waves)
static int seg_threads(int n) {
    const int t = (n + kSegRows - 1) / kSegRows * kLineGroup;
    return (t + 63) / 64 * 64;
}
static int seg_groups(int n) { return (n * n + kLineGroup - 1) / kLineGroup; }

fpde_status launch_lod3d_batch(const Lod3DBatch& b, hipStream_t st) {
    if (b.count < 1 || b.count > kMax3DBatch) { set_error("batched 3D step: 1 to 8 solves"); return FPDE_ERR_ARG; }
    int T = 0;                                            // threads of the longest lines' segments
    for (int j = 0; j < b.count; j++) {
        if (!lateral3d_partitioned(b.row[j].n, b.row[j].L)) {
            set_error("batched 3D step: partitioned sweeps only (n <= 128)");
            return FPDE_ERR_ARG;
        }
        T = std::max(T, seg_threads(b.row[j].n));
    }
    const int gn = b.first_node[b.count], gl = b.first_line[b.count];
    // the lateral sweeps evaluate their coefficients themselves (rows' Kl, iCl null)
    hipLaunchKernelGGL(k_hist_combine_batch, dim3(gn), dim3(256), 0, st, b);
    hipLaunchKernelGGL(k_lateral3d_batch, dim3(gl), dim3(T), 0, st, b, 2);
    hipLaunchKernelGGL(k_lateral3d_batch, dim3(gl), dim3(T), 0, st, b, 1);
    hipLaunchKernelGGL(k_zline3d_batch, dim3(gl), dim3(T), 0, st, b);
    FPDE_HIP_TRY(hipGetLastError());
    return FPDE_OK;
}

fpde_status launch_series3d(double* S, double* H, int P, const double* dnew, const double* ser_c,
                            const double* ser_v, int64_t nodes, int64_t ld, double hscale, hipStream_t st) {
    hipLaunchKernelGGL(k_series3d, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, st, S, H, P, dnew, ser_c,
                       ser_v, nodes, ld, hscale);
    return FPDE_OK;
}

fpde_status launch_coef3d(const double* U, int n, double h, double ksat, int mode, double* K,
                          double* iC, hipStream_t st) {
    int64_t nn = (int64_t)n * n * n;
    hipLaunchKernelGGL(k_coef3d, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, U, n, h, ksat, mode, K, iC);
    return FPDE_OK;
}

fpde_status launch_lateral3d(const double* Uin, double* Uout, const double* K, const double* iC, const double* H, int n,
                             int axis, double h2inv, double L, double* Al, double* Bt, double kap,
                             const double* E, double h, double ksat, int mode, hipStream_t st) {
    int nl = n * n;
    if (lateral3d_partitioned(n, L)) {
        hipLaunchKernelGGL(k_lateral3d_seg, dim3(seg_groups(n)), dim3(seg_threads(n)), 0, st, Uin, Uout, K, iC, H, n,
                           axis, h2inv, L, kap, E, h, ksat, mode);
        return FPDE_OK;
    }
    if (!K || !iC) { set_error("3D lateral sweep over 128 nodes needs the coefficient pass"); return FPDE_ERR_ARG; }
    hipLaunchKernelGGL(k_lateral3d, dim3((nl + 255) / 256), dim3(256), 0, st, Uin, Uout, K, iC, H, n, axis, h2inv, L,
                       Al, Bt, kap, E);
    return FPDE_OK;
}

fpde_status launch_zline3d(const double* V, double* U, const double* utop, int n, double h, double h2inv,
                           double ksat, int mode, double L, double* Dlev, double kap, const double* E,
                           const double* K, const double* iC, const double* H, hipStream_t st) {
    if (n > 256) { set_error("3D grid: at most 256 nodes per axis"); return FPDE_ERR_ARG; }
    if (lateral3d_partitioned(n, L)) {
        hipLaunchKernelGGL(k_zline3d_seg, dim3(seg_groups(n)), dim3(seg_threads(n)), 0, st, V, U, utop, n, h, h2inv,
                           ksat, mode, L, Dlev, kap, E, K, iC, H);
        return FPDE_OK;
    }
    int bs = ((n + 63) / 64) * 64;
    hipLaunchKernelGGL(k_zline3d, dim3(n * n), dim3(bs), 0, st, V, U, utop, n, h, h2inv, ksat, mode, L, Dlev, kap, E,
                       H);
    return FPDE_OK;
}

fpde_status launch_hist_combine(double* S, const Hist3D& h, int64_t nodes, double hscale, hipStream_t st) {
    hipLaunchKernelGGL(k_hist_combine, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, st, S, h, nodes, hscale);
    return FPDE_OK;
}

fpde_status launch_fold3d(const Fold3DBatch& b, hipStream_t st) {
    if (b.count < 1) return FPDE_OK;
    for (int j = 0; j < b.count; j++) {
        const int len = b.row[j].len;
        if (len != 8 && len != 16 && (len < 32 || len % 32)) { set_error("3D fold: 8, 16 or whole 32 levels"); return FPDE_ERR_ARG; }
    }
    hipLaunchKernelGGL(k_fold3d, dim3(b.first[b.count]), dim3(256), 0, st, b);
    return FPDE_OK;
}

}  // namespace fpde
