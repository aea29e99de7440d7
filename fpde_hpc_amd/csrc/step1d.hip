// One launch of the 1D implicit FP64 step (gfx950).
//
// The reference step (fpde_hpc_1d.cpp:4672-4725: al1, Om1, bt1, back
// substitution) is a Thomas sweep over the whole line; on the GPU a single
// sequential sweep of 1e4 rows is latency bound, so the line is cut into C
// chunks of <= 256 nodes, one workgroup each (partitioned / SPIKE-style
// solve):
//  - a chunk's first node s is its separator; the rows after it are solved by
//    one wave for three right-hand sides, giving U_i = x_i + y_i U_s + z_i U_s'
//    in terms of the separators s and s' (the next chunk's);
//  - the separators' rows, with the chunks put in, form a tridiagonal system of
//    C rows, which every workgroup solves redundantly before it substitutes
//    back.
// The separators' values pass between the workgroups through an exchange in
// memory within one cooperative launch, or from one launch to the next
// (k_step1d: one launch per Picard iteration and no grid-wide barrier).
// Rows (fpde_hpc_1d.cpp:3095-3142 with Dg=1, gamma=1):
//   A_i U_{i-1} - R_i U_i + B_i U_{i+1} = Om_i,
//   A_i = K_{i-1}/C_i/h^2, B_i = K_i/C_i/h^2, R_i = (K_i+K_{i-1})/C_i/h^2 + L,
//   Om_i = -L U^n_i + S_n[i]      (Om1, :4165-4268; S_n = Da*history sum)
// row 0: Dirichlet U_0 = u_top; row N-1: zero flux U_{N-1} = U_{N-2}
// (al1/bt1 with the bottom formula of U1, :4684-4703, bcN()=0).
#include "fpde_internal.h"

namespace fpde {

// Far partial sums plus the near levels t in [near_lo, t_end) of step n: the
// partial rows and levels in batches of independent loads (up to 32 partial
// rows in one memory round trip, a sum over m levels in ~m/32).  omega is read
// only at n-t-1 >= 1.
__device__ inline double hist_row(const Step1DArgs& g, int i, int n, int near_lo, int t_end, int nsplit,
                                  const double* __restrict__ part, const double* __restrict__ omega) {
    constexpr int W = 32;
    double far = 0.0;
    part += i;
    auto rows = [&](int r0, auto width) {          // (rows past the last: the last again, not added)
        constexpr int V = decltype(width)::value;
        double v[V];
#pragma unroll
        for (int j = 0; j < V; j++) v[j] = part[(int64_t)min(r0 + j, nsplit - 1) * g.part_stride];
#pragma unroll
        for (int j = 0; j < V; j++) far += r0 + j < nsplit ? v[j] : 0.0;
    };
    if (nsplit == 1) far = *part;
    else if (nsplit > 0 && nsplit <= 8) rows(0, std::integral_constant<int, 8>{});
    else
        for (int r0 = 0; r0 < nsplit; r0 += W) rows(r0, std::integral_constant<int, W>{});
    double nr0 = 0.0, nr1 = 0.0;
    for (int t0 = near_lo; t0 < t_end; t0 += W) {
        double v[W], w[W];
#pragma unroll
        for (int j = 0; j < W; j++) {
            int t = t0 + j;
            bool ok = t < t_end;
            v[j] = ok ? g.D[(int64_t)t * g.ld + i] : 0.0;
            w[j] = ok ? omega[n - t - 1] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < W; j += 2) {
            nr0 = fma(w[j], v[j], nr0);
            nr1 = fma(w[j + 1], v[j + 1], nr1);
        }
    }
    return far + (nr0 + nr1);
}

// The history of step n in memory, all levels but the newest (which the caller
// adds): the row of the levels t < n-2, summed here or ahead by the previous
// step's launch, and level n-2.
__device__ inline double hist_mem(const Step1DArgs& g, int i, int n, int64_t part_off,
                                  const double* __restrict__ omega) {
    const bool last = g.near_lo <= n - 2;
    double v = 0.0, w = 0.0;
    if (last) { v = g.D[(int64_t)(n - 2) * g.ld + i]; w = omega[1]; }
    return fma(w, v, hist_row(g, i, n, g.near_lo, n - 2, g.nsplit, g.part + part_off, omega));
}

// The newest level and the two-level corrections of the oldest intervals,
// written with explicit fma so that every kernel rounds them alike:
// om0 dnew + corr[2n] d0 + corr[2n+1] d1, with d0 = dnew at n = 1 and
// d1 = dnew at n = 2.
// c0 = corr[2n], c1 = corr[2n+1].
__device__ inline double hist_tail(double om0, double c0, double c1, int n, int near_lo, double dnew, double d0m,
                                   double d1m) {
    const double w0 = (near_lo <= n - 1) ? om0 : 0.0;
    double cr = (n == 1) ? c0 * dnew : c0 * (n >= 2 ? d0m : 0.0);
    if (n == 2) cr = fma(c1, dnew, cr);
    else if (n >= 3) cr = fma(c1, d1m, cr);
    return fma(w0, dnew, cr);
}

// ---------------------------------------------------------------------------
// Cooperative form: one launch runs the steps [n, n_end) of a history block
// with every Picard iteration inside, all C chunk workgroups co-resident.
// A workgroup has RW row waves (one thread per chunk node: coefficients, rows
// and the node's history) and one solver wave (the chunk's line solve, the
// grid exchange, the reduced system).  Per Picard iteration:
//   row waves    K and 1/C at the iterate (the solver wave: K of the node left
//                of the chunk), row data to LDS                    -- barrier A
//   solver wave  chunk rows -> U_i = x_i + y_i U_s + z_i U_s', the separators
//                s (the chunk's first node) and s' (the next chunk's);
//                publishes 7 values and the chunk's measure; waits for every
//                chunk's; decides convergence the reference way (stop once
//                max|U^k - U^{k-1}| <= tol, the iterate U^k is the result);
//                solves the C separators' system; U of its nodes to LDS
//   row waves    meanwhile: the next step's history from memory    -- barrier B
// A step's history needs only the workgroup's own nodes (its own earlier
// writes of D) and the precomputed far partials, so steps follow each other
// without a barrier; U and D of every step are written as in the
// per-iteration launches.
//
// What bounds it: the dependent chain of one iteration (coefficients, line
// solve, one grid exchange), not memory or arithmetic.  So the line solve sits
// in ONE wave: 64 lanes of R rows each, the lane's interior rows eliminated in
// registers, then parallel cyclic reduction over the 64 lanes with no
// workgroup barrier and (from stride 4 on) no LDS either, since lane
// 16 (p mod 4) + p/4 holds position p and a stride of 4 q positions is a DPP
// row shift by q.  One separator per chunk (not both chunk ends) halves the
// reduced system, whose couplings fall off with the chunk length: its cyclic
// reduction ends as soon as none exceeds kNoCoupling.
// Measured (cycles of one iteration at N = 10^4, 53 chunks, phase timers): row
// waves 2000 from barrier to barrier (coefficients 640); solver wave: rows and
// line solve 2500, publishing 900, waiting for the other chunks 4700,
// decision 150, separators 1100, U to LDS 500.  Headline solve (N = 10^4, M =
// 2 10^4) 200 ms, N = 1000, M = 2000 19.7 ms, six N = 10^4, M = 2000 in a batch
// 25.3 ms; 374, 34.2 and 57.8 ms with the whole workgroup's cyclic reduction over
// LDS, both chunk ends as separators (five words per row and level, a workgroup
// barrier per level), coefficients by square roots and divisions (1700 cycles)
// and the far parts' K splits added between the launches.
//
// The arithmetic is written with explicit fma and contraction off: single
// and batched launches round alike in every instantiation.

// Grid exchange: the 8 values a chunk publishes per barrier travel as sixteen
// 64-bit words in one 128-byte line, each holding one 32-bit half of a double
// and the 32-bit tag of the barrier it belongs to (xtag | (barrier index + 1)
// mod 2^16; xtag carries the launch count in its upper 16 bits, never 0).
// Words are written and read with relaxed agent-scope atomics: each is
// single-copy atomic and coherent across the XCDs, and a reader takes a word
// once it carries the barrier's tag, so it holds that barrier's value.  No
// fence orders one word against another, so a barrier needs no L2 write-back
// or invalidate.  The writer stores its line by one instruction (lanes 0..15),
// readers load four chunks' lines per instruction and transpose through LDS.
//  - Words alternate by barrier parity.  A workgroup writes barrier b+1's
//    words only after it has read every workgroup's barrier-b words, and each
//    workgroup wrote those after reading its barrier-(b-1) words, so no word
//    is overwritten while a reader still needs it.
//  - At launch start each workgroup zeroes its own words (no tag is 0), so no
//    word an earlier launch left can carry one of this launch's tags.
//  - A reader waits at most `wait_ticks` ticks of the device's constant wall
//    clock per wait (the host sizes it to 2 s): workgroups of a cooperative
//    launch can become resident late when other streams' kernels hold CUs at
//    dispatch, which ends within micro- to milliseconds; the bound exists so
//    that a launch whose workgroups can never all be resident ends with an
//    error instead of hanging.
// Values of chunk j: 0..3 its separator's row with the chunk's own interior
// eliminated (coupling to the node left of it, diagonal, coupling to the next
// separator, right-hand side), 4..6 x, y, z of its last node, 7 its measure.
constexpr int kXchWords = 16;                                   // per chunk and parity
constexpr int kXchMeasure = 14;                                 // first word of value 7
constexpr int kXchPad = kXchWords + 2;                          // LDS row: 144 B, 16-byte reads spread over the banks
static_assert(2 * kMaxChunks * kXchWords * 8 == (int)kXchBytes, "exchange buffer size");

// Coupling of two separators (or positions) that is dropped: its part of the one
// is below rounding, 2^-53, where the other is up to 2^20 times as large, which
// is the range of heads from 1e-2 to 1e4 m.  (At 2^-60 a dry separator of 1e6
// beside wet nodes of 1e-2 lost 3e-12 of them.)  Comparing the parts with the
// values themselves cost 1% of a solve on its dependent chain and 4% of the plain
// form's, whether the neighbours' values were fetched or bounded over the wave;
// 2^-86, another level of reduction for 32 orders at N = 4000, 4% of that solve.
constexpr double kNoCoupling = 0x1p-73;

// ---- one wave's line solve -------------------------------------------------
// a double moved within the rows of 16 lanes; lanes without a source take fill
template <int CTRL>
__device__ inline double dpp_fill(double v, double fill) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(fill), __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(fill), __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

__device__ inline int lane_of(int p) { return 16 * (p & 3) + (p >> 2); }

// The value of v at position p + OFF (p: this lane's); fill outside 0..63.
template <int OFF>
__device__ inline double at_offset(double v, int p, double fill) {
    if constexpr (OFF % 4 == 0) {
        constexpr int Q = OFF / 4;
        if constexpr (Q > 0) return dpp_fill<0x100 + Q>(v, fill);          // row_shl: from lane + Q
        else return dpp_fill<0x110 - Q>(v, fill);                          // row_shr: from lane - |Q|
    } else {
        const int q = p + OFF;
        const int src = lane_of(q & 63) << 2;
        const int lo = __builtin_amdgcn_ds_bpermute(src, __double2loint(v));
        const int hi = __builtin_amdgcn_ds_bpermute(src, __double2hiint(v));
        return (q >= 0 && q < 64) ? __hiloint2double(hi, lo) : fill;
    }
}

// One level of cyclic reduction over the 64 positions (rows a x_{p-S} + x_p +
// c x_{p+S} = d).  Past the ends stand the boundary values UL and UR: there a
// and c stay couplings to them (the partner row "x = U").
template <int S>
__device__ inline void pcr_level(double& a, double& c, double& d, int p) {
#pragma clang fp contract(off)
    const double am = at_offset<-S>(a, p, -1.0), cm = at_offset<-S>(c, p, 0.0), dm = at_offset<-S>(d, p, 0.0);
    const double ap = at_offset<S>(a, p, 0.0), cp = at_offset<S>(c, p, -1.0), dp = at_offset<S>(d, p, 0.0);
    const double inv = rcp_nr(fma(-c, ap, fma(-a, cm, 1.0)));
    d = fma(-c, dp, fma(-a, dm, d)) * inv;
    a = -(a * am) * inv;
    c = -(c * cp) * inv;
}

// Whether some row still couples to a row S positions away (NaN counts).
template <int S>
__device__ inline bool coupled(double a, double c, int p) {
    const bool l = p >= S && !(fabs(a) <= kNoCoupling), r = p + S < 64 && !(fabs(c) <= kNoCoupling);
    return __any(l || r);
}

// Solve the 64 R rows a x_{i-1} + x_i + c x_{i+1} = d of one wave (position p
// holds rows R p .. R p + R-1) between the boundary values UL (left of row 0)
// and UR (right of the last): x_i = x + y UL + z UR.  A position's first R-1
// rows are eliminated against its last one (Thomas with both couplings as
// right-hand sides), the last ones reduced cyclically.  With EARLY the
// reduction stops once no coupling between positions exceeds kNoCoupling (the
// boundaries' couplings must be zero: y and z are not formed).
template <int R, bool EARLY>
__device__ inline void wave_line(const double (&a)[R], const double (&c)[R], const double (&d)[R], int p,
                                 double (&x)[R], double (&y)[R], double (&z)[R]) {
#pragma clang fp contract(off)
    double A = a[R - 1], Cc = c[R - 1], Dd = d[R - 1];
    if constexpr (R > 1) {
        double q[R];                               // c' of the elimination
        x[0] = d[0];
        y[0] = -a[0];
        q[0] = c[0];
#pragma unroll
        for (int j = 1; j < R - 1; j++) {
            const double inv = rcp_nr(fma(-a[j], q[j - 1], 1.0));
            q[j] = c[j] * inv;
            x[j] = fma(-a[j], x[j - 1], d[j]) * inv;
            y[j] = -(a[j] * y[j - 1]) * inv;
        }
        z[R - 2] = -q[R - 2];
#pragma unroll
        for (int j = R - 3; j >= 0; j--) {
            x[j] = fma(-q[j], x[j + 1], x[j]);
            y[j] = fma(-q[j], y[j + 1], y[j]);
            z[j] = -(q[j] * z[j + 1]);
        }
        // the position's last row: its left neighbour and the next position's first row put in
        const double xn = at_offset<1>(x[0], p, 0.0), yn = at_offset<1>(y[0], p, 0.0), zn = at_offset<1>(z[0], p, 1.0);
        const double inv = rcp_nr(fma(Cc, yn, fma(A, z[R - 2], 1.0)));
        Dd = fma(-Cc, xn, fma(-A, x[R - 2], Dd)) * inv;
        A = (A * y[R - 2]) * inv;
        Cc = (Cc * zn) * inv;
    }
    // (the last position's c goes to UR)
    if constexpr (EARLY) {
        if (coupled<1>(A, Cc, p)) {
            pcr_level<1>(A, Cc, Dd, p);
            if (coupled<2>(A, Cc, p)) {
                pcr_level<2>(A, Cc, Dd, p);
                if (coupled<4>(A, Cc, p)) {
                    pcr_level<4>(A, Cc, Dd, p);
                    if (coupled<8>(A, Cc, p)) {
                        pcr_level<8>(A, Cc, Dd, p);
                        if (coupled<16>(A, Cc, p)) {
                            pcr_level<16>(A, Cc, Dd, p);
                            if (coupled<32>(A, Cc, p)) pcr_level<32>(A, Cc, Dd, p);
                        }
                    }
                }
            }
        }
        x[R - 1] = Dd;
        y[R - 1] = z[R - 1] = 0.0;
        if constexpr (R > 1) {
            const double xl = at_offset<-1>(Dd, p, 0.0);
#pragma unroll
            for (int j = 0; j < R - 1; j++) x[j] = fma(z[j], Dd, fma(y[j], xl, x[j]));
        }
    } else {
        pcr_level<1>(A, Cc, Dd, p);
        pcr_level<2>(A, Cc, Dd, p);
        pcr_level<4>(A, Cc, Dd, p);
        pcr_level<8>(A, Cc, Dd, p);
        pcr_level<16>(A, Cc, Dd, p);
        pcr_level<32>(A, Cc, Dd, p);
        x[R - 1] = Dd;
        y[R - 1] = -A;
        z[R - 1] = -Cc;
        if constexpr (R > 1) {
            // the left neighbour position's last row (row 0's: UL itself)
            const double xl = at_offset<-1>(x[R - 1], p, 0.0), yl = at_offset<-1>(y[R - 1], p, 1.0),
                         zl = at_offset<-1>(z[R - 1], p, 0.0);
#pragma unroll
            for (int j = 0; j < R - 1; j++) {
                const double y0 = y[j], z0 = z[j];
                x[j] = fma(z0, x[R - 1], fma(y0, xl, x[j]));
                y[j] = fma(z0, y[R - 1], y0 * yl);
                z[j] = fma(z0, z[R - 1], y0 * zl);
            }
        }
    }
}

// Row `row` of a solved line in every lane (row is uniform).
template <int R>
__device__ inline double line_value(const double (&x)[R], int row) {
    double v = x[0];
#pragma unroll
    for (int j = 1; j < R; j++) {
        double t = x[j];
        asm("" : "+v"(t));                          // a select of values, not of places in an array in memory
        v = (row % R == j) ? t : v;
    }
    const int l = __builtin_amdgcn_readfirstlane(lane_of(row / R));
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// LDS operations of one wave complete in order; these keep the compiler from
// moving them across a hand-over between lanes
__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kRows = 256;                                      // nodes per chunk at most
// position of chunk row r in the LDS row arrays: one double of padding per 32
// keeps the solver wave's reads at stride R doubles free of bank conflicts
__device__ inline int row_slot(int r) { return r + (r >> 5); }
constexpr int kRowSlots = kRows + 1 + (kRows >> 5) + 1;

struct Step1DLds {
    double K[kRowSlots], iC[kRowSlots], d[kRowSlots], u[kRowSlots];
    double pub[8];
    double weights[4][128];                                     // per row wave: of a fold or a near field
    alignas(16) unsigned long long words[kMaxChunks * kXchPad];
    int status;
};

enum { kNoCheck = 0, kCheckMet, kCheckPending, kDecide };         // what an exchange decides
enum { kSolved = 0, kMet, kNotMet, kRollback, kTimeout };         // and what came of it

// Value k of chunk j from its words in LDS.
__device__ inline double xch_value(const Step1DLds& L, int j, int k) {
    const ulonglong2 w = *reinterpret_cast<const ulonglong2*>(&L.words[j * kXchPad + 2 * k]);
    return __longlong_as_double((long long)((w.y << 32) | (w.x & 0xffffffffull)));
}

// The separators' system: RR rows per lane, row r of it from chunk r's values
// 0..3 in v[..][0..3] and the left chunk's 4..6 in v[..][4..6] (any finite
// values for a row without one).  Returns the values at the separators c-1, c
// and c+1 (0 past the ends).
template <int RR>
__device__ inline void solve_separators(const double (&v)[RR][7], int C, int c, int p, double& xm, double& x0,
                                        double& xp) {
#pragma clang fp contract(off)
    double a[RR], cc[RR], d[RR], x[RR], y[RR], z[RR];
#pragma unroll
    for (int j = 0; j < RR; j++) {
        const int r = RR * p + j;
        const bool ok = r < C;
        // (row 0 has v0 = 0: the values read for a left neighbour, its own chunk's, do not enter)
        const double inv = rcp_nr(fma(v[j][0], v[j][6], v[j][1]));
        a[j] = ok ? (v[j][0] * v[j][5]) * inv : 0.0;
        cc[j] = ok && r + 1 < C ? v[j][2] * inv : 0.0;
        d[j] = ok ? fma(-v[j][0], v[j][4], v[j][3]) * inv : 0.0;
    }
    wave_line<RR, true>(a, cc, d, p, x, y, z);
    xm = c > 0 ? line_value<RR>(x, c - 1) : 0.0;
    x0 = line_value<RR>(x, c);
    xp = c + 1 < C ? line_value<RR>(x, c + 1) : 0.0;
}

template <int RR>
__device__ inline void separator_rows(const Step1DLds& L, int C, int p, double (&v)[RR][7]) {
#pragma unroll
    for (int j = 0; j < RR; j++) {
        const int r = RR * p + j, rr = r < C ? r : 0, rl = rr > 0 ? rr - 1 : 0;
#pragma unroll
        for (int k = 0; k < 7; k++) v[j][k] = xch_value(L, k < 4 ? rr : rl, k);
    }
}

// One wave's elimination of a chunk: interior rows s+1 .. e (ni of them, R per
// lane) from the chunk's K, 1/C and right-hand sides in LDS; U_i = x + y U_s +
// z U_s' with the separators s and s'.  Values 0..6 of the chunk to pub.  Kh:
// K at node s-1.
template <int R>
__device__ __forceinline__ void chunk_line(const double* K, const double* iC, const double* dr, int N, int s, int ni,
                                           int c, int p, double Kh, double Ln, double h2inv, double (&x)[R],
                                           double (&y)[R], double (&z)[R], double* pub) {
#pragma clang fp contract(off)
    const int r0 = R * p;
    double a[R], cc[R], d[R];
    double Kv[R + 1], iv[R], dv[R];
#pragma unroll
    for (int j = 0; j <= R; j++) Kv[j] = K[row_slot(r0 + j)];
#pragma unroll
    for (int j = 0; j < R; j++) { iv[j] = iC[row_slot(r0 + 1 + j)]; dv[j] = dr[row_slot(r0 + 1 + j)]; }
    const double K0 = K[0], i0 = iC[0], d0 = dr[0];
#pragma unroll
    for (int j = 0; j < R; j++) {
        const double Km = Kv[j], Kp = Kv[j + 1];
        const double inv = rcp_nr(-fma(iv[j], Kp * h2inv + Km * h2inv, Ln));
        a[j] = Km * iv[j] * h2inv * inv;
        cc[j] = Kp * iv[j] * h2inv * inv;
        d[j] = dv[j] * inv;
        // bottom row U_{N-1} = U_{N-2}; rows past the chunk hand on the next
        // separator's value: x_q = x_{q+1}
        const bool in = r0 + j < ni, bottom = r0 + j == N - 2 - s;
        a[j] = in ? (bottom ? -1.0 : a[j]) : 0.0;
        cc[j] = in ? (bottom ? 0.0 : cc[j]) : -1.0;
        d[j] = in && !bottom ? d[j] : 0.0;
    }
    // the separator's row (node 0: U = u_top)
    const double as = c > 0 ? Kh * i0 * h2inv : 0.0;
    const double cs = c > 0 ? K0 * i0 * h2inv : 0.0;
    const double bs = c > 0 ? -fma(i0, K0 * h2inv + Kh * h2inv, Ln) : 1.0;
    wave_line<R, false>(a, cc, d, p, x, y, z);
    if (p == 0) {
        pub[0] = as;
        pub[1] = fma(cs, y[0], bs);
        pub[2] = cs * z[0];
        pub[3] = fma(-cs, x[0], d0);
    }
    // the last node's row: which of the lane's R is launch-uniform
    double xl = x[0], yl = y[0], zl = z[0];
#pragma unroll
    for (int j = 1; j < R; j++) {
        const bool is = (ni - 1) % R == j;
        xl = is ? x[j] : xl;
        yl = is ? y[j] : yl;
        zl = is ? z[j] : zl;
    }
    if (p == (ni - 1) / R) {
        pub[4] = xl;
        pub[5] = yl;
        pub[6] = zl;
    }
}

// ---------------------------------------------------------------------------
// Per-iteration form (plain history, space-fractional scheme, step_mode 1,
// captured steps): one launch is [finish the previous solve] + [history term,
// coefficients, rows, chunk elimination of this solve].  The chunks' values of
// the separators' system (red: per launch parity, 8 doubles per chunk: 0..6 as
// in the exchange above, 7 the chunk's max |U^k - U^{k-1}|) are written by one
// launch and solved by every wave of the next, redundantly and without a
// barrier; the nodes' x, y, z stay in xyz for its back-substitution.  The
// launch order stands in for the grid barrier.
// What bounds it: the dependent chain again (one memory trip, the separators,
// the coefficients, one barrier, the line in wave 0), so it has the cooperative
// form's wave-level solves: at N = 3001 a launch takes 7.8 us against 11.8 us
// with the whole workgroup's cyclic reduction over LDS and both chunk ends as
// separators.  Workgroups past the chunks stream the next step's plain history
// meanwhile, 16 levels in flight per thread; with them, and the partial rows
// and last levels loaded in one trip, the launch takes 7.3 us and no launch of
// the stream (4.4 us) stands between two steps.  SPACE: the space-fractional
// scheme (compiled apart: its code in the other form cost 9% of the step).
template <int RW, int RR, bool SPACE>
__global__ __launch_bounds__(64 * RW) void k_step1d(Step1DArgs g) {
#pragma clang fp contract(off)
    __shared__ double sK[kRowSlots], sC[kRowSlots], sR[kRowSlots], pub[8], wmax[RW];
    __shared__ double sKh;
    constexpr int T = 64 * RW;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int p = 4 * (lane & 15) + (lane >> 4);
    const int c = blockIdx.x;
    const int N = g.N, C = g.C;
    const int n = g.n;
    if (c >= C) {                         // the next step's history
        __shared__ double wwin[kPlainWin];
        const int b = c - C;
        if (g.ahead_splits == 0) {
            const int j = b * T + tid;
            if (j < N) g.ahead_part[j] = hist_row(g, j, n + 1, g.ahead_lo, n - 1, g.ahead_rows, g.ahead_far, g.ahead_omega);
            return;
        }
        plain_stream<T, 16>(g.D + (int64_t)g.ahead_lo * g.ld, g.ld, N, g.n + 1 - g.ahead_lo, g.ahead_hi - g.ahead_lo,
                            g.ahead_chunk, g.omega, g.ahead_part, b % g.ahead_tiles, b / g.ahead_tiles, wwin);
        return;
    }
    const int s = (int)(((int64_t)c * N) / C);
    const int nc = (int)(((int64_t)(c + 1) * N) / C) - s;
    const int i = s + tid;
    const bool act = tid < nc;
    const bool first = g.k <= 0;          // first Picard iteration of step n (or finalize)

    // ---- 0. loads that do not depend on the pending solve (one round trip) ---
    const double* const red = g.red + (size_t)(1 - g.parity) * C * 8;
    double v[RR][7], dprev = 0.0, xh = 0.0, yh = 0.0, zh = 0.0;   // h: node s-1 of the chunk to the left
    // Picard convergence of the previous launch (decided one launch late: the
    // test needs the max over every chunk): the measures it left and the
    // iterate it stored
    const bool check_conv = g.recover && g.prev_k >= 1;
    if (g.recover) {
#pragma unroll
        for (int j = 0; j < RR; j++) {
            const int r = RR * p + j, rr = r < C ? r : 0, rl = rr > 0 ? rr - 1 : 0;
#pragma unroll
            for (int k = 0; k < 7; k++) v[j][k] = red[8 * (k < 4 ? rr : rl) + k];
            if (check_conv) dprev = fmax(dprev, red[8 * rr + 7]);
        }
        if (c > 0) { xh = red[8 * c - 4]; yh = red[8 * c - 3]; zh = red[8 * c - 2]; }
    }
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (g.recover && act && tid > 0) { fx = g.xyz[i]; fy = g.xyz[g.ld + i]; fz = g.xyz[2 * g.ld + i]; }
    double uold = act ? g.U[i] : 0.0;                    // U^{n-1} (recovering, k=0) or U^n
    double Sk = (!first && act) ? g.Sbuf[i] : 0.0;
    const bool series = g.ser_P > 0;
    const int64_t drow = series ? ((n - 1) & 1) : (n - 1);    // row of D[n-1]
    double dmem = (first && !g.recover && act && n >= 1) ? g.D[drow * g.ld + i] : 0.0;
    double d0m = (first && !series && act && n >= 2) ? g.D[i] : 0.0;
    double d1m = (first && !series && act && n >= 3) ? g.D[g.ld + i] : 0.0;
    // previous iterate: the initial one for iteration 1, else the stored one
    double uitp = 0.0;
    if ((check_conv || g.k >= 1) && act) uitp = (g.k == 1) ? g.Uit0[i] : g.Uit[i];
    // halo node s-1 (owned by chunk c-1, whose workgroup rewrites U and D in
    // this launch): the converged iterate and U^{n-1} come from buffers that
    // no workgroup writes in this launch; on a thread without a node of its
    // own when there is one (else thread 0 does both evaluations)
    const int halo_tid = (nc < T) ? T - 1 : 0;
    const bool halo = tid == halo_tid && c > 0;
    const bool extrap0 = first && g.k == 0 && g.extrap && n >= 1;
    double uit_halo = (halo && check_conv) ? g.Uit[s - 1] : 0.0;
    double u_halo = (halo && !g.recover) ? g.U[s - 1] : 0.0;
    double uprev_halo = (halo && extrap0) ? g.uend[(size_t)((n - 1) & 1) * 2 * C + 2 * c - 1] : 0.0;
    double hm = (first && !series && g.k == 0 && act && n >= 1) ? hist_mem(g, i, n, g.part_off, g.omega) : 0.0;

    // space-fractional scheme: Om1's explicit sum -inv_dw_dh E_i (:4182-4189);
    // E of step n is formed by its first launch and reused by the others
    double E = 0.0;
    if (SPACE && g.k >= 0 && i > 0 && i < N - 1 && act) {
        E = first ? space_sum(g.sp_P, g.sp_ldp, g.sp_corr, g.sp_F, i) : g.sp_E[i];
        if (first) g.sp_E[i] = E;
    }

    // ---- 1. finish the previous solve: separators, then back-substitute ------
    double val = 0.0, um = 0.0, us = 0.0, up = 0.0;
    bool conv = false;
    if (g.recover) {
        solve_separators<RR>(v, C, c, p, um, us, up);
        val = tid == 0 ? us : fma(fz, up, fma(fy, us, fx));
        // node s-1 as its own chunk forms it (a chunk of one node: its separator)
        u_halo = fma(zh, us, fma(yh, um, xh));
        // the previous Picard iterate met the tolerance: it is the step's result
        if (check_conv) conv = wave_max(dprev) <= g.tol;
        if (conv) { val = uitp; u_halo = uit_halo; }
    }

    // ---- 2. advance the state -----------------------------------------------
    double un = 0.0, uit = 0.0, S = 0.0;
    if (first) {
        if (act) {
            un = uold;
            double dnew = dmem;
            if (g.recover) {                     // val = U^n, uold = U^{n-1}
                dnew = val - uold;
                g.D[drow * g.ld + i] = dnew;
                g.U[i] = val;
                un = val;
            }
            if (g.k >= 0 && n >= 1 && series) {
                // moments += newest interval, then the series (sum_alg 2)
                S = series_update(g.H, g.ld, i, g.ser_P, dnew, g.ser_c, g.ser_v);
            } else if (g.k >= 0 && n >= 1) {
                // S_n = far + near (in memory) + newest level + two-level corrections
                S = hm + hist_tail(g.omega[0], g.corr[2 * n], g.corr[2 * n + 1], n, g.near_lo, dnew, d0m, d1m);
            }
            if (g.k >= 0) g.Sbuf[i] = S;
            // Picard starts from the extrapolation 2 U^n - U^{n-1}; the
            // iterate is kept for the convergence test of the next launch and
            // the chunk ends of U^n for the next step's halo
            uit = un;
            if (g.extrap && g.k == 0) {
                if (n >= 1) uit = un + dnew;
                g.Uit0[i] = uit;
                double* ue = g.uend + (size_t)(n & 1) * 2 * C;
                if (tid == nc - 1) ue[2 * c + 1] = un;
            }
        }
    } else if (act) {
        un = uold;
        S = Sk;
        uit = val;
    }
    if (g.k < 0) {                               // finalize only (uniform)
        // space-fractional scheme: F of U^n for this chunk's rows (Om1
        // equation 0, fpde_hpc_1d.cpp:4176-4179), the arithmetic of
        // k_space_flux.  The neighbours s-1 and e+1 come from the separators
        // (or the converged iterate), so the next step needs no flux launch.
        if (SPACE && g.recover) {
            double* sU = sR;                     // U^n of nodes s-1 .. e+1
            double* sKf = sK;                    // K at U^n of nodes s-1 .. e
            double k, icv;
            if (act) {
                vgm_coefs(un, i * g.h, g.ksat, g.coef_mode, k, icv);
                sU[tid + 1] = un;
                sKf[tid + 1] = k;
            }
            if (tid == halo_tid) {
                if (c > 0) {
                    vgm_coefs(u_halo, (s - 1) * g.h, g.ksat, g.coef_mode, k, icv);
                    sU[0] = u_halo;
                    sKf[0] = k;
                }
                if (c < C - 1) sU[nc + 1] = conv ? g.Uit[s + nc] : up;
            }
            __syncthreads();
            if (act) {
                double f = 0.0;
                if (i >= 1 && i <= N - 2) {
                    const double ul = sU[tid], u0 = sU[tid + 1], ur = sU[tid + 2];
                    const double Km = sKf[tid], Kj = sKf[tid + 1];
                    f = space_flux(Km, Kj, ul, u0, ur, g.h);
                }
                g.sp_F[i] = f;
            }
        }
        return;
    }

    double* const mine = g.red + ((size_t)g.parity * C + c) * 8;
    if (!first && conv) {
        // converged: hand the iterate on unchanged, x = U, y = z = 0 and the
        // separator's row "U_s = U" (measure 0 keeps later launches of this
        // step passing it on)
        if (act && tid > 0) { g.xyz[i] = uit; g.xyz[g.ld + i] = 0.0; g.xyz[2 * g.ld + i] = 0.0; }
        if (tid == 0) { mine[0] = 0.0; mine[1] = 1.0; mine[2] = 0.0; mine[3] = uit; mine[7] = 0.0; }
        if (tid == nc - 1) { mine[4] = uit; mine[5] = 0.0; mine[6] = 0.0; }
        return;                                  // uniform: every wave forms conv alike
    }
    if (!first) {
        // |U^{k} - U^{k-1}| over the chunk; U^0 of the step is the initial
        // iterate stored by the k = 0 launch
        const double d = wave_max(act ? fabs(uit - uitp) : 0.0);
        if (lane == 0) wmax[wave] = d;
        if (act) g.Uit[i] = uit;
    }

    // ---- 3. coefficients at the iterate, right-hand sides -------------------
    // (space-fractional scheme: the diffusion part of A_/B/R scaled by
    // Dg kb(gamma,i-1,i,i))
    const double kap = SPACE ? g.sp_kap : 1.0;
    if (extrap0) u_halo += u_halo - uprev_halo;
    const bool spare = halo && !act;             // (in the same evaluation as the wave's own nodes)
    double K, invC;
    vgm_coefs(spare ? u_halo : uit, (spare ? s - 1 : i) * g.h, g.ksat, g.coef_mode, K, invC);
    if (spare) sKh = K * kap;
    if (act) {
        const int slot = row_slot(tid);
        sK[slot] = K * kap;
        sC[slot] = invC;
        sR[slot] = i == 0 ? g.utop : fma(-invC, E, fma(-g.L, un, S));
    }
    if (halo && act) {
        vgm_coefs(u_halo, (s - 1) * g.h, g.ksat, g.coef_mode, K, invC);
        sKh = K * kap;
    }
    __syncthreads();
    if (wave > 0) return;

    // ---- 4. the chunk's elimination, in wave 0 ------------------------------
    double x[RW], y[RW], z[RW];
    chunk_line<RW>(sK, sC, sR, N, s, nc - 1, c, p, c > 0 ? sKh : 0.0, g.L, g.h2inv, x, y, z, pub);
    double* const to = g.xyz + s + 1 + RW * p;
#pragma unroll
    for (int j = 0; j < RW; j++)
        if (RW * p + j < nc - 1) { to[j] = x[j]; to[g.ld + j] = y[j]; to[2 * g.ld + j] = z[j]; }
    if (p == 0) {
        double d = 0.0;
        if (!first)
#pragma unroll
            for (int w = 0; w < RW; w++) d = fmax(d, wmax[w]);
        pub[7] = d;
    }
    wave_lds_sync();
    if (lane < 8) mine[lane] = pub[lane];
}

// Where a launch stands: step n, Picard iteration k of it, and what the next
// exchange decides.  Both roles of a workgroup run it on the same results, so
// it stays uniform.  A step whose last Picard iteration is due (k =
// picard_max - 1) ends tentatively with U^k when the launch has a next step:
// its convergence measure goes out with the next step's first iteration, so
// the exchange that decides it is the one that carries those rows.  If it did
// not converge, every workgroup restores the step, runs its last iteration,
// rewrites D[n] and U, and starts the next step again.  Series moments are
// updated in place, so sum_alg 2 decides convergence before the step ends.
enum { kGoOn = 0, kStepEnds, kStepEndsTentatively, kGoBack, kLeave };
struct PicardState {
    int n, n_end, k, check, picard_max, solves;
    bool pending, redo, tentative_ok;
    __device__ inline void begin(int n_, bool pending_) {
        n = n_;
        k = 0;
        redo = false;
        pending = pending_;
        check = pending ? kCheckPending : kNoCheck;
    }
    __device__ inline int after(int st) {
        if (st == kSolved) {
            solves++;
            k++;
            pending = false;
            if (redo || k == picard_max) return kStepEnds;
            const bool due = k == picard_max - 1;
            if (due && tentative_ok && n + 1 < n_end) return kStepEndsTentatively;
            check = due ? kDecide : kCheckMet;     // (due: decided before the last iteration, which it may save)
            return kGoOn;
        }
        if (st == kNotMet) { check = kNoCheck; return kGoOn; }
        return st == kMet ? kStepEnds : (st == kRollback ? kGoBack : kLeave);
    }
    __device__ inline void back(int n_) {          // to the last iteration of step n_
        n = n_;
        redo = true;
        pending = false;
        check = kNoCheck;
    }
};

__device__ inline PicardState picard_state(const Step1DArgs& g) {
    PicardState ps{};
    ps.n_end = g.n_end;
    ps.picard_max = g.picard_max;
    ps.tentative_ok = g.ser_P == 0;
    ps.begin(g.n, false);
    return ps;
}

// s_waitcnt vmcnt(0), the other counters left alone (loads and stores share
// vmcnt on gfx9)
constexpr int kDrainVmem = 0x0f70;

// A launch constant kept in vector registers (the two roles have more of them
// than scalar registers, and a spilled scalar costs two moves per use).
__device__ inline double in_vgpr(double v) { asm("" : "+v"(v)); return v; }

// Steps [g.n, g.n_end) of one solve by its chunk workgroup c (0 <= c < g.C):
// a row wave.  Each thread keeps NPT nodes of the chunk, 64 RW apart.
template <int RW, int NPT>
__device__ __forceinline__ void row_steps(const Step1DArgs& g, const int c, Step1DLds& L) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x;
    const int s = (int)(((int64_t)c * g.N) / g.C);
    const int nc = (int)(((int64_t)(c + 1) * g.N) / g.C) - s;
    const bool series = g.ser_P > 0;
    const double ksat = in_vgpr(g.ksat), L0 = in_vgpr(g.L), utop = in_vgpr(g.utop);
    auto row = [&](int q) { return tid + 64 * RW * q; };       // this thread's chunk rows
    auto act = [&](int q) { return row(q) < nc; };

    // state carried from step to step: U^n and D[n-1] of the node (from
    // memory at the first step of the launch)
    const int n_first = g.n;
    double zi[NPT], un[NPT], dlast[NPT], d0m[NPT], d1m[NPT];
    double* const Dc = g.D + s + min(tid, nc - 1);             // the first node's column of D (idle threads: the last node's)
    auto level = [&](int q, int m) { return Dc + 64 * RW * q + (int64_t)(series ? (m & 1) : m) * g.ld; };
#pragma unroll
    for (int q = 0; q < NPT; q++) {
        const bool ok = act(q);
        zi[q] = in_vgpr((s + row(q)) * g.h);
        un[q] = ok ? g.U[s + row(q)] : 0.0;
        dlast[q] = (ok && n_first >= 1) ? *level(q, n_first - 1) : 0.0;
        // D[0], D[1] (corrections of the two oldest intervals): from memory
        // when written by an earlier launch, else taken when this launch
        // makes them
        d0m[q] = (!series && ok && n_first >= 1) ? *level(q, 0) : 0.0;
        d1m[q] = (!series && ok && n_first >= 2) ? *level(q, 1) : 0.0;
    }
    // Near-field groups folded ahead into g.mid: group j (levels near_lo + 16 j
    // ...+15) is final, whatever the pending decision on the previous step,
    // from step s_j = near_lo + 16 j + 17 on (levels t <= s_j - 2; n0 if that
    // is later).  The first iteration of step s_j + b folds it for the 8 steps
    // from s_j + 2 + 8 b on, so a fold is spread over the steps that follow
    // (done at once for a whole block it stalled the chain: 56 dependent
    // batches per 128-step block), and step m's history, formed at step m - 1,
    // finds every group with s_j < m - 1 and sums the other levels itself (at
    // most 17; near_lo is n0 or up to 31 levels before it).  The schedule
    // depends on the step alone: launches may end anywhere in a block.
    auto ready = [&](int j) { return max(g.n0, g.near_lo + kNearGroup * j + kNearGroup + 1); };    // s_j
    auto groups = [&](int m) { return m - 2 >= g.n0 ? (m - 3 - g.near_lo) / kNearGroup : 0; };
    int fold_done = n_first - 1;                               // (a step done again does not fold again)
    PicardState ps = picard_state(g);
    // of a tentatively ended step, what its last iteration still needs
    double sv_un[NPT], sv_S[NPT];
    // the in-memory part of the history sum (far partials and near levels
    // t < n) and the tail weights omega[0], corr[2n], corr[2n+1]: of this step
    // and of the next one (formed beside this step's first line solve)
    double hm[NPT], hm_next[NPT];
    double w0 = 0.0, w1 = 0.0, w2 = 0.0, w0_next = 0.0, w1_next = 0.0, w2_next = 0.0;
    double S[NPT], it[NPT];
    // local coefficient: one, or the step's own (prescribed grid)
    double Ln = g.Lv ? g.Lv[n_first] : L0, Ln_prev = Ln, Ln_next = Ln;
#pragma unroll
    for (int q = 0; q < NPT; q++) sv_un[q] = sv_S[q] = hm[q] = hm_next[q] = 0.0;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    double* const wl = L.weights[wave];
    // step m's history from memory (levels t < m - 1).  Every load of a node
    // goes out before the first is used (one memory round trip), the weights
    // once per wave, through LDS.
    auto history = [&](int m, double (&h)[NPT], double& a0, double& a1, double& a2) {
        const double* om = g.omega + (int64_t)(m - g.n0) * g.omega_stride;
        a0 = om[0];
        a1 = g.corr[2 * m];
        a2 = g.corr[2 * m + 1];
        const int folded = groups(m);
        const int lo = g.near_lo + kNearGroup * folded;
        constexpr int W = 16;
        wl[lane] = om[1 + min(lane, max(m - 2 - lo, 0))];      // wl[k]: weight of level m - 2 - k
        wave_lds_sync();
#pragma unroll
        for (int q = 0; q < NPT; q++) {
            const int col = act(q) ? 64 * RW * q : 0;          // (idle threads read a column that exists)
            const double* pt = g.part + (int64_t)(m - g.n0) * g.ld + (Dc - g.D) + col;
            const double* d = Dc + (int64_t)lo * g.ld + col;
            constexpr int F = 5;                               // partial rows loaded together
            double v[W], f[F], md = 0.0;
#pragma unroll
            for (int j = 0; j < W; j++) {
                v[j] = 0.0;
                if (lo + j < m - 1) v[j] = *d;
                d += g.ld;
                asm("" : "+v"(d));                             // (one running address)
            }
#pragma unroll
            for (int k = 0; k < F; k++) {
                f[k] = 0.0;
                if (k < g.nsplit) f[k] = *pt;
                pt += g.part_stride;
                asm("" : "+v"(pt));
            }
            if (folded > 0) md = g.mid[(int64_t)(m - g.n0) * g.ld + (Dc - g.D) + col];
            double far = f[0] + f[1];
#pragma unroll
            for (int k = 2; k < F; k++) far += f[k];
            for (int k = F; k < g.nsplit; k++) { far += *pt; pt += g.part_stride; }
            double n0 = md, n1 = 0.0;
#pragma unroll
            for (int j = 0; j < W; j += 2) {
                n0 = fma(wl[max(m - 2 - lo - j, 0)], v[j], n0);
                n1 = fma(wl[max(m - 3 - lo - j, 0)], v[j + 1], n1);
            }
            // levels past the first 16: a 17th, and those before a block's first two steps
            for (int t = lo + W; t < m - 1; t++) n0 = fma(om[m - 1 - t], Dc[(int64_t)t * g.ld + col], n0);
            h[q] = far + (n0 + n1);
        }
        wave_lds_sync();
    };
    // group j of 16 levels into g.mid for the steps [p0, p1), p1 - p0 <= 8
    auto fold = [&](int j, int p0, int p1) {
        const int lo = g.near_lo + kNearGroup * j;
        // weight of level lo + k at step p0 + r: wl[16 r + k]
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int q = lane + 64 * h, pr = min(p0 + (q >> 4), p1 - 1);
            wl[q] = g.omega[(int64_t)(pr - g.n0) * g.omega_stride + pr - lo - 1 - (q & 15)];
        }
        wave_lds_sync();
#pragma unroll 1
        for (int q = 0; q < NPT; q++) {
            if (!act(q)) break;
            double dv[kNearGroup], acc[kFoldBatch];
            const double* d = Dc + (int64_t)lo * g.ld + 64 * RW * q;
            double* mp = g.mid + (int64_t)(p0 - g.n0) * g.ld + (Dc - g.D) + 64 * RW * q;
            const double* mr = mp;
#pragma unroll
            for (int k = 0; k < kNearGroup; k++) {
                dv[k] = *d;
                d += g.ld;
                asm("" : "+v"(d));
            }
#pragma unroll
            for (int r = 0; r < kFoldBatch; r++) {
                acc[r] = 0.0;
                if (j > 0 && p0 + r < p1) acc[r] = *mr;
                mr += g.ld;
                asm("" : "+v"(mr));
            }
#pragma unroll
            for (int r = 0; r < kFoldBatch; r++) {
#pragma unroll
                for (int k = 0; k < kNearGroup; k++) acc[r] = fma(wl[16 * r + k], dv[k], acc[r]);
                if (p0 + r < p1) *mp = acc[r];
                mp += g.ld;
                asm("" : "+v"(mp));
            }
        }
        wave_lds_sync();
    };
    auto start_step = [&]() {
        const int n = ps.n;
#pragma unroll
        for (int q = 0; q < NPT; q++) {
            S[q] = 0.0;
            if (n >= 1 && act(q))
                S[q] = series ? series_update(g.H, g.ld, s + row(q), g.ser_P, dlast[q], g.ser_c + (size_t)n * g.ser_P,
                                              g.ser_v + (size_t)n * g.ser_P)
                              : hm[q] + hist_tail(w0, w1, w2, n, g.near_lo, dlast[q], d0m[q], d1m[q]);
            // Picard starts from 2 U^n - U^{n-1} (a single pass: lagged at U^n)
            it[q] = (g.extrap && n >= 1) ? un[q] + dlast[q] : un[q];
        }
    };
    if (!series && n_first >= 1) history(n_first, hm, w0, w1, w2);
    start_step();
    bool fresh = true;                                         // the step's first iteration
    __builtin_amdgcn_s_waitcnt(kDrainVmem);
    for (;;) {
        if (ps.check != kDecide) {
#pragma unroll
            for (int q = 0; q < NPT; q++) {
                double K, invC;
                vgm_coefs(it[q], zi[q], ksat, g.coef_mode, K, invC);
                if (act(q)) {
                    const int slot = row_slot(row(q));
                    L.K[slot] = K;
                    L.iC[slot] = invC;
                    L.d[slot] = s + row(q) == 0 ? utop : fma(-Ln, un[q], S[q]);
                }
            }
        }
        __syncthreads();                                       // A
        if (fresh && !series) {
            if (ps.n > fold_done) {
                fold_done = ps.n;
                for (int j = 0; j < groups(ps.n + 2); j++) {
                    const int p0 = ready(j) + 2 + kFoldBatch * (ps.n - ready(j)), end = g.n0 + g.blk;
                    if (p0 < end) fold(j, p0, min(p0 + kFoldBatch, end));
                }
            }
            // the next step's history from memory (levels t < n are written;
            // D[n] enters through the tail)
            if (ps.n + 1 < g.n_end) history(ps.n + 1, hm_next, w0_next, w1_next, w2_next);
        }
        if (fresh && g.Lv && ps.n + 1 < g.n_end) Ln_next = g.Lv[ps.n + 1];
        // memory drained here, beside the solver wave: from barrier B to the
        // next A only the stores of D and U are under way, and no load's wait
        // has to sit out their way to memory
        __builtin_amdgcn_s_waitcnt(kDrainVmem);
        __syncthreads();                                       // B
        double unew[NPT];
#pragma unroll
        for (int q = 0; q < NPT; q++) {
            unew[q] = L.u[row_slot(row(q))];
            asm volatile("" : "+v"(unew[q]));                  // (read beside the status, not after it)
        }
        const int st = __builtin_amdgcn_readfirstlane(L.status);
#pragma unroll
        for (int q = 0; q < NPT; q++) {
            it[q] = st == kSolved ? unew[q] : it[q];
        }
        fresh = false;
        const int what = ps.after(st);
        if (what == kGoOn) continue;
        if (what == kLeave) return;
        if (what == kGoBack) {
            // the tentatively ended step n - 1 needs its last iteration (from
            // its iterate, now in un; dlast, D[0] and D[1] are set at its end)
#pragma unroll
            for (int q = 0; q < NPT; q++) { it[q] = un[q]; un[q] = sv_un[q]; S[q] = sv_S[q]; }
            ps.back(ps.n - 1);
            Ln_next = Ln;
            Ln = Ln_prev;
            continue;
        }
        // step n is done: the last iterate is U^{n+1}
        const int n = ps.n;
        Ln_prev = Ln;
        Ln = Ln_next;
#pragma unroll
        for (int q = 0; q < NPT; q++) {
            sv_un[q] = un[q];
            sv_S[q] = S[q];
            const double dn = it[q] - un[q];
            if (act(q)) {
                *level(q, n) = dn;
                g.U[s + row(q)] = it[q];
            }
            dlast[q] = dn;
            un[q] = it[q];
            d0m[q] = n == 0 ? dn : d0m[q];                     // (unconditional: kept in registers)
            d1m[q] = n == 1 ? dn : d1m[q];
            hm[q] = ps.redo ? hm[q] : hm_next[q];
        }
        if (n + 1 == g.n_end) return;
        // (after a step done again its successor's history part is at hand)
        w0 = ps.redo ? w0 : w0_next;
        w1 = ps.redo ? w1 : w1_next;
        w2 = ps.redo ? w2 : w2_next;
        ps.begin(n + 1, what == kStepEndsTentatively);
        start_step();
        fresh = true;
    }
}

// The same steps by the solver wave: R rows per lane, 64 R > chunk nodes - 1.
// It follows the iterates of its rows and of node s-1 (whose K the
// separator's row needs), so the chunk's measure max|U^{k+1} - U^k| is formed
// here, while the row waves evaluate the coefficients.
template <int R>
__device__ __forceinline__ void solver_steps(const Step1DArgs& g, const int c, Step1DLds& L) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int N = g.N, C = g.C;
    const int s = (int)(((int64_t)c * N) / C);
    const int ni = (int)(((int64_t)(c + 1) * N) / C) - s - 1;  // interior rows s+1 .. e
    const int pos = 4 * (lane & 15) + (lane >> 4);             // this lane's position in the line solve
    const int first_row = R * pos;                             // its rows: chunk nodes first_row+1 .. first_row+R
    const bool series = g.ser_P > 0;
    const double zh = in_vgpr((s - 1) * g.h), ksat = in_vgpr(g.ksat), h2inv = in_vgpr(g.h2inv), tol = in_vgpr(g.tol);
    const double L0 = in_vgpr(g.L);
    // node r of this lane (r = R: the separator s, r = R + 1: node s-1)
    auto node = [&](int r) { return r < R ? s + 1 + first_row + r : s + R - r; };
    auto have = [&](int r) { return r < R ? first_row + r < ni : (r == R || c > 0); };
    constexpr int NV = R + 2;
    double un[NV], dlast[NV], it[NV], sv_un[NV];
    const int n_first = g.n;
#pragma unroll
    for (int r = 0; r < NV; r++) {
        un[r] = have(r) ? g.U[node(r)] : 0.0;
        dlast[r] = (have(r) && n_first >= 1)
                       ? g.D[(int64_t)(series ? ((n_first - 1) & 1) : n_first - 1) * g.ld + node(r)]
                       : 0.0;
        sv_un[r] = 0.0;
    }
    int bk = 0;                                                // grid barriers passed in this launch
    auto xbase = [&](int b) { return g.xch + (size_t)(b & 1) * kMaxChunks * kXchWords; };
    auto xtag = [&](int b) { return g.xtag | ((unsigned)(b + 1) & 0xffffu); };
    // the exchange words of this workgroup, both parities, zeroed before its
    // first publication (by the lanes that publish them)
    if (lane < kXchWords)
        for (int par = 0; par < 2; par++)
            __hip_atomic_store(xbase(par) + c * kXchWords + lane, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    auto publish = [&](int b, int lo) {                        // words lo..15 of the values in L.pub
        wave_lds_sync();
        const unsigned long long t = (unsigned long long)xtag(b) << 32;
        if (lane >= lo && lane < kXchWords)
            __hip_atomic_store(xbase(b) + c * kXchWords + lane,
                               t | reinterpret_cast<const unsigned*>(L.pub)[lane], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    };
    // whether a wait that began at *t0 (-1: now) has run out of time (the
    // launch then ends; the host reports it)
    auto timed_out = [&](int64_t* t0) -> bool {
        const int64_t now = (int64_t)wall_clock64();
        if (*t0 < 0) *t0 = now;
        if (now - *t0 <= g.wait_ticks) return false;
        __hip_atomic_store(g.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    };
    // every chunk's words into L.words once they carry the barrier's tag, 64
    // chunks per round: load k takes chunks 4 k .. 4 k + 3 of the round; the
    // largest measure on the way (its halves sit in lanes 14 and 15 of each
    // row of 16)
    auto collect = [&](int b, double& largest) -> bool {
        const unsigned tg = xtag(b);
        int64_t t0 = -1;
        constexpr int K = 16;
        for (int j0 = 0; j0 < C; j0 += 64) {
            unsigned long long w[K];
            int l = lane;
            asm volatile("" : "+v"(l));                        // (addresses formed here, not kept across iterations)
            const unsigned long long* x = xbase(b) + j0 * kXchWords + l;
            const int kn = min(K, (C - j0 + 3) >> 2);          // loads of this round
            const int mine = (C - j0 - (l >> 4) + 3) >> 2;     // and those whose chunk exists on this lane
#pragma unroll
            for (int k = 0; k < K; k++) {
                w[k] = 0;
                if (k < kn) w[k] = __hip_atomic_load(x + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            for (;;) {
                unsigned miss = 0;
#pragma unroll
                for (int k = 0; k < K; k++) miss |= k < mine ? (unsigned)(w[k] >> 32) ^ tg : 0u;
                if (__all(miss == 0)) break;
                if (timed_out(&t0)) return false;
#pragma unroll
                for (int k = 0; k < K; k++)
                    if (k < mine && (unsigned)(w[k] >> 32) != tg)
                        w[k] = __hip_atomic_load(x + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            unsigned long long* to = &L.words[(j0 + (l >> 4)) * kXchPad + (l & 15)];
            double m = 0.0;
#pragma unroll
            for (int k = 0; k < K; k++) {
                if (k < mine) to[4 * k * kXchPad] = w[k];
                // lane 15 of a row: its own half above lane 14's
                const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)w[k], 0x111, 0xf, 0xf, false);
                m = fmax(m, k < mine ? __hiloint2double((int)(unsigned)w[k], lo) : 0.0);
            }
#pragma unroll
            for (int r = 15; r < 64; r += 16)
                largest = fmax(largest, __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(m), r),
                                                         __builtin_amdgcn_readlane(__double2loint(m), r)));
        }
        wave_lds_sync();
        return true;
    };
    // the measure words alone
    auto collect_measures = [&](int b, double& largest) -> bool {
        const unsigned tg = xtag(b);
        int64_t t0 = -1;
        for (int j0 = 0; j0 < C; j0 += 64) {
            const int j = min(j0 + lane, C - 1);
            const unsigned long long* x = xbase(b) + j * kXchWords + kXchMeasure;
            unsigned long long w[2];
            for (;;) {
                for (int k = 0; k < 2; k++) w[k] = __hip_atomic_load(x + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (__all((unsigned)(w[0] >> 32) == tg && (unsigned)(w[1] >> 32) == tg)) break;
                if (timed_out(&t0)) return false;
            }
            largest = fmax(largest, wave_max(__longlong_as_double((long long)((w[1] << 32) | (w[0] & 0xffffffffull)))));
        }
        return true;
    };

    // Between the barriers of an iteration (Kh: K at node s-1, `meas`: the
    // chunk's measure): kSolved with the new iterate in
    // L.u and itn; where `check` asks for it, the decision
    // on the published measures (kCheckMet: U^k met the tolerance -> kMet;
    // kCheckPending: the tentatively ended previous step did not ->
    // kRollback; kDecide: the measure alone is exchanged -> kMet or kNotMet);
    // kTimeout when a wait ran out of time.
    auto line_solve = [&](int b, int check, double Kh, double Ln, double meas, double (&itn)[NV]) -> int {
        double x[R], y[R], z[R];
        const bool decide = check == kDecide;
        int p = pos;
        asm volatile("" : "+v"(p));                            // (addresses and masks formed here, not kept across iterations)
        const int r0 = R * p;
        if (!decide)
            chunk_line<R>(L.K, L.iC, L.d, N, s, ni, c, p, Kh, Ln, h2inv, x, y, z, L.pub);
        if (lane == 0) L.pub[7] = meas;
        publish(b, decide ? kXchMeasure : 0);
        double largest = 0.0;
        if (!(decide ? collect_measures(b, largest) : collect(b, largest))) return kTimeout;
        const bool met = __builtin_amdgcn_readfirstlane(largest <= tol ? 1 : 0) != 0;     // (uniform)
        if (decide) return met ? kMet : kNotMet;
        double um, us, up;
        const double xl = c > 0 ? xch_value(L, c - 1, 4) : 0.0, yl = c > 0 ? xch_value(L, c - 1, 5) : 0.0,
                     zl = c > 0 ? xch_value(L, c - 1, 6) : 0.0;
        if (C <= 64) {
            double v[1][7];
            separator_rows<1>(L, C, p, v);
            solve_separators<1>(v, C, c, p, um, us, up);
        } else {
            double v[4][7];
            separator_rows<4>(L, C, p, v);
            solve_separators<4>(v, C, c, p, um, us, up);
        }
        if (check == kCheckMet && met) return kMet;
        if (check == kCheckPending && !met) return kRollback;
#pragma unroll
        for (int j = 0; j < R; j++) {
            itn[j] = fma(z[j], up, fma(y[j], us, x[j]));
            L.u[row_slot(r0 + 1 + j)] = itn[j];
        }
        if (lane == 0) L.u[0] = us;
        itn[R] = us;
        itn[R + 1] = fma(zl, us, fma(yl, um, xl));             // node s-1 as its own chunk forms it
        return kSolved;
    };

    PicardState ps = picard_state(g);
    double Ln = 0.0, meas = 0.0;                               // meas: the chunk's measure of the last solve
    auto start_step = [&]() {
        Ln = g.Lv ? g.Lv[ps.n] : L0;
        const bool ex = g.extrap && ps.n >= 1;
#pragma unroll
        for (int r = 0; r < NV; r++) it[r] = ex ? un[r] + dlast[r] : un[r];
    };
    start_step();
    for (;;) {
        double Kh, iCh;
        vgm_coefs(it[R + 1], zh, ksat, g.coef_mode, Kh, iCh);
        __syncthreads();                                       // A
        double itn[NV];
        const int st = __builtin_amdgcn_readfirstlane(line_solve(bk, ps.check, Kh, Ln, meas, itn));
        if (lane == 0) L.status = st;
        __syncthreads();                                       // B
        bk++;
        if (st == kSolved) {
            double change = 0.0;
#pragma unroll
            for (int r = 0; r < NV; r++) {
                if (r <= R) change = fmax(change, have(r) ? fabs(itn[r] - it[r]) : 0.0);
                it[r] = itn[r];
            }
            meas = wave_max(change);                           // (beside the row waves' coefficients)
        }
        const int what = ps.after(st);
        if (what == kGoOn) continue;
        if (what == kLeave) return;
        if (what == kGoBack) {
#pragma unroll
            for (int r = 0; r < NV; r++) { it[r] = un[r]; un[r] = sv_un[r]; }
            ps.back(ps.n - 1);
            Ln = g.Lv ? g.Lv[ps.n] : L0;
            continue;
        }
        const int n = ps.n;
#pragma unroll
        for (int r = 0; r < NV; r++) { sv_un[r] = un[r]; dlast[r] = it[r] - un[r]; un[r] = it[r]; }
        if (n + 1 == g.n_end) break;
        ps.begin(n + 1, what == kStepEndsTentatively);
        start_step();
    }
    // the launch's Picard iterations, counted once per solve (err[1])
    if (c == 0 && lane == 0)
        __hip_atomic_fetch_add(g.err + 1, ps.solves, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The body of the single-solve launch and of the batched one: RW row waves of
// NPT nodes per thread, then the solver wave of RW NPT rows per lane.  The roles are compiled apart and
// keep their control flow flat: together (one loop with the role inside) their
// launch constants overflowed the scalar registers, and the reloads and
// branches between two solves cost 2500 of 15000 cycles.
template <int RW, int NPT>
__global__ __launch_bounds__(64 * RW + 64) void k_step1d_block(Step1DArgs g) {
    __shared__ Step1DLds L;
    if (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) == RW) solver_steps<RW * NPT>(g, (int)blockIdx.x, L);
    else row_steps<RW, NPT>(g, (int)blockIdx.x, L);
}

// Many independent solves in one cooperative launch: workgroups
// [t.first[j], t.first[j+1]) are the chunks of solve j.  Each solve keeps its
// own exchange words, measures and Picard decisions, so its arithmetic
// is that of its single-solve launch; the fields that change from block to
// block come with the launch, the rest from the solve's row of `base`.  Two
// row waves of two nodes per thread and the solver wave (whose rows per lane
// are those of the single-solve launch): two workgroups share a CU at 256
// registers per lane, so a batch holds up to 512 chunk workgroups, and their
// latency-bound waves interleave on each SIMD.
constexpr int kBatchThreads = 192;
__global__ __launch_bounds__(kBatchThreads, 2) void k_step1d_batch(const Step1DArgs* __restrict__ base, BatchTick t) {
    __shared__ Step1DLds L;
    const int wg = (int)blockIdx.x;
    int j = 0;
    while (j + 1 < t.count && wg >= t.first[j + 1]) j++;
    Step1DArgs g = base[j];
    g.n = t.n[j];
    g.n_end = t.n_end[j];
    g.n0 = t.n0[j];
    g.nsplit = t.nsplit[j];
    g.near_lo = t.near_lo[j];
    g.xtag = t.xtag[j];
    g.part_stride = t.part_stride[j];
    g.part = t.part[j];
    const int c = wg - t.first[j];
    if (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) < 2) row_steps<2, 2>(g, c, L);
    else if (row_waves(g.N, g.C) == 3) solver_steps<3>(g, c, L);
    else solver_steps<4>(g, c, L);
}

// Barrier bound in wall-clock ticks: 2 s at the device's wall clock rate
// (hipDeviceAttributeWallClockRate, kHz).
int64_t barrier_wait_ticks() {
    int dev = 0, khz = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
        khz = 100000;                                  // the 100 MHz constant clock of gfx9 parts
    return (int64_t)khz * 2000;
}

static bool coop_fits(const void* kern, int threads, int64_t wgs) {
    int dev = 0, coop = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !coop) return false;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return false;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, threads, 0) != hipSuccess) return false;
    return (int64_t)per_cu * cus >= wgs;
}

// Chunks of up to 192 nodes: three row waves; longer ones four, or two with two
// nodes per thread (slim).
struct BlockKernel { const void* fn; int threads; };
static BlockKernel block_kernel(int N, int C, bool slim) {
    if (row_waves(N, C) == 3) return {(const void*)k_step1d_block<3, 1>, 256};
    if (slim) return {(const void*)k_step1d_block<2, 2>, 192};
    return {(const void*)k_step1d_block<4, 1>, 320};
}

// Five waves of 247 registers put two on one SIMD of their CU and leave it no
// room for another kernel's: where the chunks cover most of the GPU, the far
// part ahead (lookahead) waits for the end of the launch it was to run beside.
// FP64 takes long enough for that to count; there the launch has the batch's
// shape, which leaves every SIMD half its registers.  Lagged / Picard, ms, five
// waves against three: N = 65536, 3000 steps 64 / 44 and 95 / 74 (57 and 101 with
// the whole workgroup's line solve in four waves), N = 55000, 2000 steps (215
// chunks) 33 / 26 and 50 / 45; N = 40000 in 157 chunks 21.2 / 21.1 and 36.5 / 38.1.
// bf16, N = 55000: 20.2 / 21.8 and 38.0 / 40.2.
bool step1d_block_slim(int N, int C) {
    int dev = 0, cus = 0;
    return row_waves(N, C) == 4 && hipGetDevice(&dev) == hipSuccess &&
           hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && 4 * C > 3 * cus;
}

// Whether the C workgroups of a cooperative block launch can be co-resident.
bool step1d_block_supported(int N, int C) {
    const BlockKernel k = block_kernel(N, C, false);
    return coop_fits(k.fn, k.threads, C);
}
bool step1d_batch_supported(int64_t wgs) { return coop_fits((const void*)k_step1d_batch, kBatchThreads, wgs); }

fpde_status launch_step1d_batch(const Step1DArgs* base, const BatchTick& t, hipStream_t st) {
    if (t.count < 1 || t.count > kMaxBatch) { set_error("batched step: 1 to 32 solves"); return FPDE_ERR_ARG; }
    for (int j = 0; j < t.count; j++)
        if (t.first[j + 1] < t.first[j]) { set_error("batched step: bad workgroup table"); return FPDE_ERR_ARG; }
    const int wgs = t.first[t.count];
    if (wgs == 0) return FPDE_OK;
    const Step1DArgs* b = base;
    BatchTick tick = t;
    void* params[] = {&b, &tick};
    FPDE_HIP_TRY(hipLaunchCooperativeKernel((const void*)k_step1d_batch, dim3(wgs), dim3(kBatchThreads), params, 0, st));
    return FPDE_OK;
}

fpde_status launch_step1d_block(const Step1DArgs& a, hipStream_t st) {
    if (a.C > kMaxChunks || (a.N + a.C - 1) / a.C > kRows) {
        set_error("1D line too long for the reduced system (N <= 65536)");
        return FPDE_ERR_ARG;
    }
    if (a.sp_on) { set_error("cooperative step: the space-fractional sum runs with per-iteration launches"); return FPDE_ERR_ARG; }
    if (a.n_end <= a.n) return FPDE_OK;
    Step1DArgs arg = a;
    void* params[] = {&arg};
    const BlockKernel k = block_kernel(a.N, a.C, a.slim != 0);
    FPDE_HIP_TRY(hipLaunchCooperativeKernel(k.fn, dim3(a.C), dim3(k.threads), params, 0, st));
    return FPDE_OK;
}

fpde_status launch_step1d(const Step1DArgs& a, hipStream_t st) {
    if (a.C > kMaxChunks || (a.N + a.C - 1) / a.C > kRows) {
        set_error("1D line too long for the reduced system (N <= 65536)");
        return FPDE_ERR_ARG;
    }
    const bool three = row_waves(a.N, a.C) == 3, few = a.C <= 64;
    auto* const kern = a.sp_on ? (three ? (few ? k_step1d<3, 1, true> : k_step1d<3, 4, true>)
                                        : (few ? k_step1d<4, 1, true> : k_step1d<4, 4, true>))
                               : (three ? (few ? k_step1d<3, 1, false> : k_step1d<3, 4, false>)
                                        : (few ? k_step1d<4, 1, false> : k_step1d<4, 4, false>));
    Step1DArgs arg = a;
    const int T = three ? 192 : 256;
    arg.ahead_tiles = (a.N + 2 * T - 1) / (2 * T);
    const int more = a.ahead_splits > 0 ? arg.ahead_tiles * a.ahead_splits : (a.ahead_part ? (a.N + T - 1) / T : 0);
    hipLaunchKernelGGL(kern, dim3(a.C + more), dim3(T), 0, st, arg);
    return FPDE_OK;
}

}  // namespace fpde
