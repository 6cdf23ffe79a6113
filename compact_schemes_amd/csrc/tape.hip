// tape.hip -- the adjoint of the fused Euler RK4 step as transposed line
// sweeps, and the forward step that records what the adjoint reads (no
// reference counterpart).
//
// For the inviscid right-hand side R(q) = sum_a [ D_a F^a(q) + C^a(q) ]
// (operators described in vjp.hip),
//   R'(q)^T t = sum_a [ (dF^a/dq)^T D_a^T (t + S_a^T mu_a) + G_a ],
// with D_a^T = B_a^T A_a^-T.  One sweep per axis evaluates, line by line:
// the seed t plus the face seeds mu_a at the two face rows; the solve with
// the LU factors of A^T (the chunked recurrences of the forward sweeps on the
// transposed table); the transposed explicit stencil B^T (inside the line the
// derivative stencil with the opposite sign, plus the closure or seam rows at
// the line ends); and the transposed flux Jacobian at every point,
// accumulated over the three sweeps.  The last sweep of a stage also carries
// the RK4 recurrence.  The filter's transpose is a sweep of the same form
// (A^T solve, then B^T) on closure lines; on cyclic lines the filter is a
// symmetric circulant and is its own transpose.  mu_a and G_a, the adjoint
// of the characteristic BC at the face points, come from a small face kernel
// that runs before the sweeps of a stage.
//
// Tape of one step: the stage states q0..q3 and, for every stage, the
// boundary derivatives of the flux divergence along each axis (what the
// characteristic BC linearises about), [4 stages][3 axes][2 face][5][face].
#include "fused_kernels.hpp"
#include "vjp_parts.hpp"

namespace cs {
namespace fused {

namespace {

// g = (dF^AX/dq)^T nu for the inviscid flux row of flux_row(): with
// ss = m (u_AX + uf) and p = (gamma-1)(E - |m|^2/(2 rho)),
//   F_0 = rho ss, F_1+i = (rho u_i) ss + [i = AX] m p, F_4 = (E + p) ss - p uf m,
// the products collect into cs (the coefficient of d ss) and cp (of d p).
template <int AX>
__device__ __forceinline__ void flux_jt(const double* q, const double* nu, double m, double uf, double* g) {
    const Prim p = primitive(q);
    const double vel = AX == 0 ? p.u : (AX == 1 ? p.v : p.w);
    const double ss = m * (vel + uf);
    const double cs = nu[1] * q[1] + nu[2] * q[2] + nu[3] * q[3] + nu[4] * (q[4] + p.p);
    const double cp = m * nu[1 + AX] + nu[4] * (m * vel);
    const double u[3] = {p.u, p.v, p.w};
    g[0] = nu[0] * (m * uf) - cs * (m * vel * p.rhoi) + cp * (kGamm1 * 0.5 * (p.u * p.u + p.v * p.v + p.w * p.w));
#pragma unroll
    for (int i = 0; i < 3; i++) g[1 + i] = nu[1 + i] * ss - cp * (kGamm1 * u[i]);
    g[1 + AX] += nu[0] * m + cs * (m * p.rhoi);
    g[4] = nu[4] * ss + cp * kGamm1;
}

// the same for a general metric row m (curvilinear grids): ss = m.(u + uf),
// F_1+i = (rho u_i) ss + m_i p, F_4 = (E + p) ss - p (uf.m); with mu = m.u,
//   g_0 = nu_0 (m.uf) - cs mu / rho + cp (gamma-1)|u|^2/2,
//   g_1+i = nu_1+i ss + nu_0 m_i + cs m_i / rho - cp (gamma-1) u_i,
//   g_4 = nu_4 ss + cp (gamma-1),
// cs = nu_1..3 . (rho u) + nu_4 (E + p), cp = nu_1..3 . m + nu_4 mu
__device__ __forceinline__ void flux_jt_m(const double* q, const double* nu, const double* m, cs_point umf,
                                          double* g) {
    const Prim p = primitive(q);
    const double u[3] = {p.u, p.v, p.w};
    const double mu = m[0] * p.u + m[1] * p.v + m[2] * p.w;
    const double mf = m[0] * umf.x + m[1] * umf.y + m[2] * umf.z;
    const double ss = m[0] * (p.u + umf.x) + m[1] * (p.v + umf.y) + m[2] * (p.w + umf.z);
    const double cs = nu[1] * q[1] + nu[2] * q[2] + nu[3] * q[3] + nu[4] * (q[4] + p.p);
    const double cp = m[0] * nu[1] + m[1] * nu[2] + m[2] * nu[3] + nu[4] * mu;
    g[0] = nu[0] * mf - cs * (mu * p.rhoi) + cp * (kGamm1 * 0.5 * (p.u * p.u + p.v * p.v + p.w * p.w));
#pragma unroll
    for (int i = 0; i < 3; i++) g[1 + i] = nu[1 + i] * ss + nu[0] * m[i] + cs * (m[i] * p.rhoi) - cp * (kGamm1 * u[i]);
    g[4] = nu[4] * ss + cp * kGamm1;
}

// AT: the transposed flux-divergence sweep along AX of one stage.
// MODE 0: gout = J^T nu (+ G); 1: gout = gin + J^T nu (+ G); 2 (last sweep of
// stages 4..2): tn = -ck (gin + J^T nu + G), tout = tn, lam += tn; 3 (last
// sweep of stage 1): lam += -ck (gin + J^T nu + G)
// CURV: the point's metric row (curvilinear solvers; their per-point
// Jacobian scales the seed before the stage, see backward_fused)
template <int AX, int MODE, bool CURV = false>
struct AT {
    static constexpr int NF = 5;
    static constexpr bool kFilter = false;
    static constexpr int kWpe = 3;        // waves per SIMD of the y/z kernels (168 VGPRs)
    // streaming rule: seed, q and the result or accumulator; lam and the next
    // seed.  MODE 1 adds in place, so its accumulator counts once (128^3 adjoint
    // 1216 -> 1166 us); MODE 3 counts as MODE 2 (40 less: 112^3 888 -> 896)
    static constexpr int kBytes = 120 + (MODE > 1 ? 80 : 0) + (CURV ? 24 : 0);
    const double* q[5];       // the stage state the RHS was evaluated at
    const double* t[5];       // seed
    const double* gin[5];
    double* gout[5];
    double* lam[5];
    double* tout[5];
    const double* mu;         // [2 face][5][nface] face seeds (added to the seed at the face rows), or null
    const double* G;          // the same layout, face-point terms
    long nface;
    double ck;
    double m, uf;
    cs_point umf;
    Metric mt;
    template <bool NT>
    __device__ __forceinline__ void seed(uoff bo, double* v) const {
#pragma unroll
        for (int f = 0; f < 5; f++) v[f] = ldg<NT>(t[f], bo);
    }
    __device__ __forceinline__ void face_seed(int face, long line, double* v) const {
        if (!mu) return;
#pragma unroll
        for (int f = 0; f < 5; f++) v[f] += mu[(face * 5 + f) * nface + line];
    }
    // what a point's result needs (loads only), the result from it and nu (in
    // d; face: 0, 1 at a face point, else -1), and its stores: the kernels
    // issue the loads of the next rows before a row's stores, which may alias
    // them for all the compiler knows
    struct Out {
        double q[5];
        double g[MODE > 0 ? 5 : 1], l[MODE > 1 ? 5 : 1], m[CURV ? 3 : 1];
    };
    template <bool NT>
    __device__ __forceinline__ void load_out(uoff bo, Out& e) const {
#pragma unroll
        for (int v = 0; v < 5; v++) e.q[v] = ldg<NT>(q[v], bo);
        if constexpr (MODE > 0) {
#pragma unroll
            for (int v = 0; v < 5; v++) e.g[v] = ldg<NT>(gin[v], bo);
        }
        if constexpr (MODE > 1) {
#pragma unroll
            for (int v = 0; v < 5; v++) e.l[v] = ldg<NT>(lam[v], bo);
        }
        if constexpr (CURV) {
#pragma unroll
            for (int k = 0; k < 3; k++) e.m[k] = ldg<NT>(mt.m[AX][k], bo);
        }
    }
    __device__ __forceinline__ void combine(Out& e, double* d, int face, long line) const {
        double g[5];
        const double c = ck;
        if constexpr (CURV) flux_jt_m(e.q, d, e.m, umf, g);
        else flux_jt<AX>(e.q, d, m, uf, g);
        if (G && face >= 0) {
#pragma unroll
            for (int v = 0; v < 5; v++) g[v] += G[(face * 5 + v) * nface + line];
        }
#pragma unroll
        for (int v = 0; v < 5; v++) {
            if constexpr (MODE == 0) d[v] = g[v];
            else if constexpr (MODE == 1) d[v] = e.g[v] + g[v];
            else if constexpr (MODE == 2) { d[v] = -c * (e.g[v] + g[v]); e.l[v] = e.l[v] + d[v]; }
            else d[v] = e.l[v] - c * (e.g[v] + g[v]);
        }
    }
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d, const double* l) const {
#pragma unroll
        for (int v = 0; v < 5; v++) {
            if constexpr (MODE == 2) {
                stg<NT>(tout[v], bo, d[v]);
                stg<NT>(lam[v], bo, l[v]);
            } else {
                stg<NT>(MODE == 3 ? lam[v] : gout[v], bo, d[v]);
            }
        }
    }
};

// FT: the transposed filter in place on five fields lmx apart; NF = 5 (all
// per workgroup) or 1 (blockIdx.y picks the field)
template <int NFV>
struct FT {
    static constexpr int NF = NFV;
    static constexpr bool kFilter = true;
    static constexpr int kWpe = 4;
    static constexpr int kBytes = 8 * NFV;      // in place
    double* q;
    long lmx;
    const double* an;         // the filter's coefficient sets (filter_bt)
    __device__ __forceinline__ double* field(int f) const {
        return q + (long)(NFV == 1 ? (int)blockIdx.y : f) * lmx;
    }
    template <bool NT>
    __device__ __forceinline__ void seed(uoff bo, double* v) const {
#pragma unroll
        for (int f = 0; f < NFV; f++) v[f] = ldg<NT>(field(f), bo);
    }
    __device__ __forceinline__ void face_seed(int, long, double*) const {}
    struct Out { double l[1]; };
    template <bool NT>
    __device__ __forceinline__ void load_out(uoff, Out&) const {}
    __device__ __forceinline__ void combine(Out&, double*, int, long) const {}
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d, const double*) const {
#pragma unroll
        for (int f = 0; f < NFV; f++) stg<NT>(field(f), bo, d[f]);
    }
};

// B^T of the derivative on the rows of a chunk from a window w holding rows
// s-2+u (wrapped on seam lines; `last` chunks are whole).  Rows i in [2, N-3]
// are interior rows, so column j receives B[i][j] = +bb, +aa, -aa, -bb from
// i = j-2, j-1, j+1, j+2: the same formula in every chunk with the other rows
// of the window taken as zero.  The closure rows (forward_system in
// adjoint.hip; build_system, src/cuda/kernels/numerics_device_pc.hpp:176-293)
// or the seam rows (pbci on the own side, pbco on the far side of the wrap)
// add at the ends.
template <int K>
__device__ __forceinline__ void deriv_bt(const double (&w)[K + 4], double (&o)[K], bool first, bool last, bool seam,
                                         const double* pb) {
    double v[K + 4];
#pragma unroll
    for (int u = 0; u < K + 4; u++)
        v[u] = u < 4 ? (first ? 0.0 : w[u]) : u >= K ? (last ? 0.0 : w[u]) : w[u];
#pragma unroll
    for (int t = 0; t < K; t++) o[t] = kAa * (v[t + 1] - v[t + 3]) + kBb * (v[t] - v[t + 4]);
    if (!first && !last) return;
    if (!seam) {
        if (first) {
            const double y0 = w[2], y1 = w[3];
            o[0] += kAb00 * y0 - kAb10 * y1;
            o[1] += kAb01 * y0;
            o[2] += kAb02 * y0 + kAb10 * y1;
        } else {
            const double yN1 = w[K + 1], yN2 = w[K];
            o[K - 1] += kAb10 * yN2 - kAb00 * yN1;
            o[K - 2] += -kAb01 * yN1;
            o[K - 3] += -kAb02 * yN1 - kAb10 * yN2;
        }
    } else {
        static_assert(K == kLmd, "seam columns span one 8-point chunk");
        const double* pbco = pb;              // pbco[16] | pbci[16]
        const double* pbci = pb + 2 * kLmd;
        if (first) {
            const double y0 = w[2], y1 = w[3], yN1 = w[1], yN2 = w[0];
#pragma unroll
            for (int t = 0; t < K; t++)
                o[t] += pbci[t] * y0 + pbci[kLmd + t] * y1 - pbco[t] * yN1 - pbco[kLmd + t] * yN2;
        } else {
            const double y0 = w[K + 2], y1 = w[K + 3], yN1 = w[K + 1], yN2 = w[K];
#pragma unroll
            for (int i = 0; i < K; i++)
                o[K - 1 - i] += pbco[i] * y0 + pbco[kLmd + i] * y1 - pbci[i] * yN1 - pbci[kLmd + i] * yN2;
        }
    }
}

// B^T of the closure-line filter from a window w holding rows s-5+u: row i has
// order 2*M, M = min(d, 5), d its distance from the nearer end, and is the
// identity at d = 0 (an + 6M = coefficient set M, as in filter_rhs).  Every
// chunk runs the order-10 formula with the rows next to the ends (d < 5) and
// past them taken as zero; those rows reach M columns each way, so they add in
// the end chunks and, of 8-point chunks, row d = 4 one column beyond.
template <int K>
__device__ __forceinline__ void filter_bt(const double (&w)[K + 10], double (&o)[K], int c, int P, bool whole,
                                          const double* an) {
    constexpr int H = 5;
    const bool first = c == 0, last = c == P - 1;
    // rows next to the ends in the neighbour chunk's window (K = 8: d = 3, 4)
    const bool second = K == 8 && c == 1, before = K == 8 && c == P - 2;
    double v[K + 10];
#pragma unroll
    for (int u = 0; u < K + 10; u++) {
        bool zero = false;
        if (u < 2 * H) zero |= first;
        if (u < 2) zero |= second;
        if (u >= K) zero |= last;
        if (u >= K + 8) zero |= before;
        if (u == K + 7) zero |= before && !whole;
        v[u] = zero ? 0.0 : w[u];
    }
#pragma unroll
    for (int t = 0; t < K; t++) {
        double x = an[30] * v[t + H];
#pragma unroll
        for (int m = 1; m <= 5; m++) x += 0.5 * an[30 + m] * (v[t + H + m] + v[t + H - m]);
        o[t] = x;
    }
    if (first || last) {
        // row at distance M from the end into the column at distance e
#pragma unroll
        for (int M = 0; M < H; M++) {
            const double y = first ? w[H + M] : w[K + H - 1 - M];
#pragma unroll
            for (int e = 0; e <= 2 * M && e < K; e++) {
                const int am = e < M ? M - e : e - M;
                const double cf = M == 0 ? 1.0 : am == 0 ? an[6 * M] : 0.5 * an[6 * M + am];
                if (first) o[e] += cf * y;
                else o[K - 1 - e] += cf * y;
            }
        }
    }
    if (second) o[0] += 0.5 * an[28] * w[1];
    if (before) {
        if (whole) o[K - 1] += 0.5 * an[28] * w[K + 8];
        else o[K - 2] += 0.5 * an[28] * w[K + 7];
    }
}

template <int K, class SW, int W>
__device__ __forceinline__ void stencil_t(const SW& sw, const double (&w)[W], double (&o)[K], int c, int P,
                                          bool whole, bool seam, const double* pb) {
    if constexpr (SW::kFilter) filter_bt<K>(w, o, c, P, whole, sw.an);
    else deriv_bt<K>(w, o, c == 0, c == P - 1, seam, pb);
}

constexpr int kRowsT = 2;       // rows whose epilogue loads are in flight in the y/z kernel
constexpr int kPointsT = 3;     // points of a lane in the x kernel

// ---------------------------------------------------------------------------
// transposed sweep, x lines: one wave holds the chunk groups of 64/P lines
// (a contiguous run); coalesced loads and stores, LDS transposes field by
// field, carries by wave scans.
//
// Bound by the 20 fields it reads and 10 it writes: 128^3 MODE 2 116 -> 88 us
// (5.7 TB/s), MODE 3 95 -> 73; what the y sweep left in the last-level cache
// helps.
// ---------------------------------------------------------------------------
template <int K, class SW, bool EX, bool NT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
xtT_kernel(AxisDesc ax, SweepCommon cm, SW sw) {
    constexpr int NF = SW::NF;
    constexpr int J = K;
    constexpr int H = SW::kFilter ? 5 : 2;
    constexpr int W = K + 2 * H;
    static_assert(K == 8 && H <= K, "8-point chunks; halo rows come from the neighbouring chunks only");
    extern __shared__ double lds[];       // [64/P lines][P chunks][K+1], 64 slots for lanes past the run

    const int N = ax.N, P = ax.P, NP = P * K;
    const Chunks<K, EX> ch(N, P);
    const int lane = threadIdx.x;
    const int lpw = 64 / P;
    const long line0 = group_of(ax.xcd) * lpw;
    const int nl = (int)min((long)lpw, ax.nlines - line0);
    const int npts = nl * N;
    const uoff run = line_off(0, (uoff)line0, (uoff)cm.lxi, (uoff)cm.plane);
    // lanes past the run repeat its last point: no branches around the loads
    auto off = [&](int j) { return run + (uoff)min(lane + 64 * j, npts - 1) * 8u; };

    double xq[NF][J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        double x[NF];
        sw.template seed<NT>(off(j), x);
#pragma unroll
        for (int f = 0; f < NF; f++) xq[f][j] = x[f];
    }
    int slot[J], lrw[J];                 // LDS slot; line << 10 | row
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int p = lane + 64 * j;
        // p / N by the reciprocal rounded up: exact for p < 1024, N <= 1024
        const int l = (int)(((unsigned)p * ((0x1000000u + N - 1) / (unsigned)N)) >> 24), row = p - l * N;
        int c = row >> 3, t = row & 7;
        if (!EX && row >= K) {
            const int q = row - K, cs = (q * (65536 / (K - 1) + 1)) >> 16;   // q / (K-1), exact for q < 1024
            if (q < (K - 1) * ch.D) { c = cs + 1; t = q - cs * (K - 1); }
            else { c = (row + ch.D) >> 3; t = (row + ch.D) & 7; }
        }
        slot[j] = p < npts ? xt_slot<K>(l, P, c, t) : lpw * P * (K + 1) + lane;
        lrw[j] = (l << 10) | row;
    }

    const int li = lane / P, c = lane % P;
    const bool work = li < nl;
    const int lr = work ? li : 0;
    const int s = c * K;
    const bool first = c == 0, last = c == P - 1, whole = ch.whole(c);
    const double* tab = SW::kFilter ? ax.ftab : ax.tab;

    double r[NF][K];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; j++) lds[slot[j]] = xq[f][j];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < K; t++) r[f][t] = lds[xt_slot<K>(lr, P, c, EX || t < K - 1 || whole ? t : K - 2)];
    }
    if (first || last) {
        double v[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) v[f] = first ? r[f][0] : r[f][K - 1];
        sw.face_seed(first ? 0 : 1, line0 + lr, v);
#pragma unroll
        for (int f = 0; f < NF; f++) {
            r[f][0] = first ? v[f] : r[f][0];
            r[f][K - 1] = first ? r[f][K - 1] : v[f];
        }
    }

    double carry[NF], G[NF], X[NF];
    forward_local<K, NF>(tab, NP, s, r, carry);
    scan_forward<NF>(tab[3 * NP + s + K - 1], carry, c, P, G);
    apply_carry<K, NF>(tab, 3 * NP, s, r, G);
    if constexpr (!EX) zero_padding<K, NF>(r, whole);
    backward_local<K, NF>(tab, NP, s, r, carry);
    scan_backward<NF>(tab[4 * NP + s], carry, c, P, X);
    apply_carry<K, NF>(tab, 4 * NP, s, r, X);

    const bool wrap = !SW::kFilter && ax.seam;
    const int hl = c > 0 ? c - 1 : (wrap ? P - 1 : 0);
    const int hr = c + 1 < P ? c + 1 : (wrap ? 0 : P - 1);
    const int left = xt_slot<K>(lr, P, hl, K - H) - (ch.whole(hl) ? 0 : 1);
#pragma unroll
    for (int f = 0; f < NF; f++) {
        __syncthreads();
        if (work) {
#pragma unroll
            for (int t = 0; t < K; t++) lds[xt_slot<K>(li, P, c, t)] = r[f][t];
        }
        __syncthreads();
        double w[W], right[H];
#pragma unroll
        for (int u = 0; u < H; u++) {
            w[u] = lds[left + u];
            right[u] = lds[xt_slot<K>(lr, P, hr, u)];
        }
#pragma unroll
        for (int t = 0; t < K; t++) w[t + H] = r[f][t];
        close_window<K, H, W>(w, right, whole);
        double o[K];
        stencil_t<K, SW, W>(sw, w, o, c, P, whole, ax.seam, cm.pb);
#pragma unroll
        for (int t = 0; t < K; t++) r[f][t] = o[t];
    }

    double xo[NF][J];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        __syncthreads();
        if (work) {
#pragma unroll
            for (int t = 0; t < K; t++) lds[xt_slot<K>(li, P, c, t)] = r[f][t];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; j++) xo[f][j] = lds[slot[j]];
    }
    // the loads of kPointsT points ahead of the stores
    typename SW::Out e[kPointsT];
#pragma unroll
    for (int j = 0; j < kPointsT; j++) sw.template load_out<NT>(off(j), e[j]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; j++) {
        double d[NF], l[NF];
        typename SW::Out& ej = e[j % kPointsT];
#pragma unroll
        for (int f = 0; f < NF; f++) d[f] = xo[f][j];
        const int row = lrw[j] & 1023;
        sw.combine(ej, d, row == 0 ? 0 : (row == N - 1 ? 1 : -1),
                   min(line0 + (lrw[j] >> 10), ax.nlines - 1));
#pragma unroll
        for (int f = 0; f < NF; f++) l[f] = ej.l[sizeof(ej.l) > sizeof(double) ? f : 0];
        if (j + kPointsT < J) {
            sw.template load_out<NT>(off(j + kPointsT), ej);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (lane + 64 * j < npts) sw.template store<NT>(off(j), d, l);
    }
}

// ---------------------------------------------------------------------------
// transposed sweep, y/z lines: TL lines x P chunks per workgroup, each thread
// loads and stores its own chunk rows (coalesced across the TL lines), carries
// by LDS folds, halo rows of the solution through LDS
//
// Bound by latency at three waves a SIMD, as the forward sweeps are.  What it
// spent beside that were branches: one around each row's loads for the face
// terms kept them from being in flight together, and the end chunks tested
// every tap of the stencil (128^3: flux y 88 -> 72 us, z 70 -> 66, filter y
// 84 -> 32, z 90 -> 37).
// ---------------------------------------------------------------------------
template <int K, int AX, int TL, class SW, bool EX, bool NT>
__global__ void __launch_bounds__(TL * kMaxP < 1024 ? TL * kMaxP : 1024)
__attribute__((amdgpu_waves_per_eu(SW::kWpe)))
directT_kernel(AxisDesc ax, SweepCommon cm, SW sw) {
    constexpr int NF = SW::NF;
    constexpr int H = SW::kFilter ? 5 : 2;
    constexpr int W = K + 2 * H;
    static_assert(H <= K, "halo rows come from the neighbouring chunks only");
    extern __shared__ double lds[];

    const int N = ax.N, P = ax.P, NP = P * K;
    const Chunks<K, EX> ch(N, P);
    const int lloc = threadIdx.x % TL;
    const int c = TL == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / TL) : threadIdx.x / TL;
    const long line = group_of(ax.xcd) * TL + lloc;
    const bool act = line < ax.nlines;
    const long ln = act ? line : ax.nlines - 1;
    const int s = c * K;
    const bool first = c == 0, last = c == P - 1, whole = ch.whole(c);
    const uoff st = (uoff)ax.st * 8u;
    // threads past the last line repeat it, a padding row repeats the chunk's
    // last: no branches around the loads, and nothing of theirs is stored
    const uoff cbase = line_off(AX, (uoff)ln, (uoff)cm.lxi, (uoff)cm.plane) + (uoff)ch.start(c) * st;
    auto off = [&](int t) { return cbase + (uoff)(EX || t < K - 1 || whole ? t : K - 2) * st; };
    const double* tab = SW::kFilter ? ax.ftab : ax.tab;

    double r[NF][K];
#pragma unroll
    for (int t = 0; t < K; t++) {
        double x[NF];
        sw.template seed<NT>(off(t), x);
#pragma unroll
        for (int f = 0; f < NF; f++) r[f][t] = x[f];
    }
    if (first || last) {
        double v[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) v[f] = first ? r[f][0] : r[f][K - 1];
        sw.face_seed(first ? 0 : 1, ln, v);
#pragma unroll
        for (int f = 0; f < NF; f++) {
            r[f][0] = first ? v[f] : r[f][0];
            r[f][K - 1] = first ? r[f][K - 1] : v[f];
        }
    }

    double carry[NF], G[NF], X[NF];
    forward_local<K, NF>(tab, NP, s, r, carry);
#pragma unroll
    for (int f = 0; f < NF; f++) lds[(f * P + c) * TL + lloc] = carry[f];
    __syncthreads();
    fold_forward<NF, K>(lds, tab, NP, P, TL, c, lloc, G);
    apply_carry<K, NF>(tab, 3 * NP, s, r, G);
    if constexpr (!EX) zero_padding<K, NF>(r, whole);
    backward_local<K, NF>(tab, NP, s, r, carry);
    double* xb = lds + NF * P * TL;
#pragma unroll
    for (int f = 0; f < NF; f++) xb[(f * P + c) * TL + lloc] = carry[f];
    __syncthreads();
    fold_backward<NF, K>(xb, tab, NP, P, TL, c, lloc, X);
    apply_carry<K, NF>(tab, 4 * NP, s, r, X);

    // halo rows hb[(f*2H + k)*P + c][TL]: k < H the first H rows of chunk c,
    // k >= H its last H rows (neighbours wrap on seam lines of the derivative)
    const bool wrap = !SW::kFilter && ax.seam;
    const int cl = c > 0 ? c - 1 : (wrap ? P - 1 : 0), cr = c + 1 < P ? c + 1 : (wrap ? 0 : P - 1);
    __syncthreads();                      // earlier reads of the LDS are done
#pragma unroll
    for (int f = 0; f < NF; f++) {
#pragma unroll
        for (int k = 0; k < H; k++) {
            lds[((f * 2 * H + k) * P + c) * TL + lloc] = r[f][k];
            lds[((f * 2 * H + H + k) * P + c) * TL + lloc] = whole ? r[f][K - H + k] : r[f][K - H + k - 1];
        }
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < NF; f++) {
        double w[W], right[H];
#pragma unroll
        for (int k = 0; k < H; k++) {
            w[k] = lds[((f * 2 * H + H + k) * P + cl) * TL + lloc];
            right[k] = lds[((f * 2 * H + k) * P + cr) * TL + lloc];
        }
#pragma unroll
        for (int t = 0; t < K; t++) w[t + H] = r[f][t];
        close_window<K, H, W>(w, right, whole);
        double o[K];
        stencil_t<K, SW, W>(sw, w, o, c, P, whole, ax.seam, cm.pb);
#pragma unroll
        for (int t = 0; t < K; t++) r[f][t] = o[t];
    }

    if (!act) return;
    // the loads of kRowsT rows ahead of the stores
    typename SW::Out e[kRowsT];
#pragma unroll
    for (int t = 0; t < kRowsT; t++) sw.template load_out<NT>(off(t), e[t]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < K; t++) {
        double d[NF], l[NF];
        typename SW::Out& et = e[t % kRowsT];
#pragma unroll
        for (int f = 0; f < NF; f++) d[f] = r[f][t];
        sw.combine(et, d, t == 0 && first ? 0 : (t == K - 1 && last ? 1 : -1), ln);
#pragma unroll
        for (int f = 0; f < NF; f++) l[f] = et.l[sizeof(et.l) > sizeof(double) ? f : 0];
        if (t + kRowsT < K) {
            sw.template load_out<NT>(off(t + kRowsT), et);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (EX || t < K - 1 || whole) sw.template store<NT>(off(t), d, l);
    }
}

// adjoint of the characteristic BC at the face points of axis ax (the same
// products as gcbc_vjp_kernel of vjp.hip, into face buffers): lam_f = sum of
// sbcc*lam over the kMbci rows next to the face; mu = (dc/dg)^T lam_f (added
// to the seed at the face row), G = (dc/dq)^T lam_f (added at the face
// point); drv = [2 face][5][nface] boundary derivatives of the forward sweep
__global__ void __launch_bounds__(256) face_adjoint_kernel(const double* q, const double* lam, const double* sbcc,
                                                           const double* drv, double* mu, double* G, int ax, int N,
                                                           long nface, long lxi, long plane, long st, EulerPhys ph,
                                                           long lmx, const double* cmf, const double* yaco) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 2 * nface) return;
    const int face = (int)(t / nface);
    const long f = t % nface;
    long base;
    if (ax == 0) base = f * lxi;
    else if (ax == 1) base = (f / lxi) * plane + (f % lxi);
    else base = f;
    const long pt = base + (long)(face ? N - 1 : 0) * st;
    const long dir = face ? -st : st;
    double lf[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int ii = 0; ii < kMbci; ii++) {
        const long r = pt + ii * dir;
        const double w = sbcc[r];
#pragma unroll
        for (int v = 0; v < 5; v++) lf[v] += w * lam[r + v * lmx];
    }
    double qq[5], gd[5];
#pragma unroll
    for (int v = 0; v < 5; v++) {
        qq[v] = q[pt + v * lmx];
        gd[v] = drv[((long)face * 5 + v) * nface + f];
    }
    // face normal and Jacobian: the caller's arrays (curvilinear solvers) or the constants
    double cm[3], J = ph.J;
    if (yaco) {
        for (int k = 0; k < 3; k++) cm[k] = cmf[((long)face * 3 + k) * nface + f];
        J = yaco[pt];
    } else {
        const double sg = ph.m[ax] * ph.J < 0.0 ? -1.0 : 1.0;
        for (int k = 0; k < 3; k++) cm[k] = k == ax ? sg : 0.0;
    }
    typedef Dual<5> D;
    {
        D gdd[5], cr[5];
#pragma unroll
        for (int v = 0; v < 5; v++) gdd[v] = D::seed(gd[v], v);
        face_corr_at<double, D>(face, qq, gdd, cm, J, ph.umf, cr);
        D phi(0.0);
#pragma unroll
        for (int v = 0; v < 5; v++) phi = phi + cr[v] * lf[v];
#pragma unroll
        for (int v = 0; v < 5; v++) mu[((long)face * 5 + v) * nface + f] = phi.d[v];
    }
    {
        D qd[5], gdd[5], cr[5];
#pragma unroll
        for (int v = 0; v < 5; v++) {
            qd[v] = D::seed(qq[v], v);
            gdd[v] = D(gd[v]);
        }
        face_corr_at<D, D>(face, qd, gdd, cm, J, ph.umf, cr);
        D phi(0.0);
#pragma unroll
        for (int v = 0; v < 5; v++) phi = phi + cr[v] * lf[v];
#pragma unroll
        for (int v = 0; v < 5; v++) G[((long)face * 5 + v) * nface + f] = phi.d[v];
    }
}

template <int K, int AX, int TL, class SW>
const void* direct_t(bool exact, bool nt) {
    if (exact) return nt ? (const void*)directT_kernel<K, AX, TL, SW, true, true>
                         : (const void*)directT_kernel<K, AX, TL, SW, true, false>;
    return nt ? (const void*)directT_kernel<K, AX, TL, SW, false, true>
              : (const void*)directT_kernel<K, AX, TL, SW, false, false>;
}

// transposed sweep along AX on chunks of K points: x lines one wave a
// workgroup, y/z lines 16 or 64 lines; FT<1> spreads the five fields over grid.y
template <int K, int AX, class SW>
int launch_k(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, hipStream_t s) {
    constexpr int NF = SW::NF, H = SW::kFilter ? 5 : 2;
    const unsigned gy = NF == 1 ? 5u : 1u;
    const bool exact = ax.N == ax.P * K, nt = streams<SW>(ax, cm, gy);
    if constexpr (AX == 0) {
        const int lpw = 64 / ax.P;
        const size_t lds = sizeof(double) * (lpw * ax.P * (K + 1) + 64);
        const dim3 grid((unsigned)((ax.nlines + lpw - 1) / lpw), gy);
        const void* k = exact ? (nt ? (const void*)xtT_kernel<K, SW, true, true> : (const void*)xtT_kernel<K, SW, true, false>)
                              : (nt ? (const void*)xtT_kernel<K, SW, false, true> : (const void*)xtT_kernel<K, SW, false, false>);
        return launch(k, grid, dim3(64), lds, with_runs(ax, grid.x, true, 64), cm, sw, s);
    } else {
        const int TL = SW::NF == 1 && ax.P <= 16 ? 64 : 16;      // as block_lines
        const size_t halo = (size_t)NF * 2 * H * ax.P * TL, carries = (size_t)2 * NF * ax.P * TL;
        const size_t lds = sizeof(double) * (halo > carries ? halo : carries);
        const dim3 grid((unsigned)((ax.nlines + TL - 1) / TL), gy);
        const void* k = nullptr;
        if constexpr (NF == 1)
            if (TL == 64) k = direct_t<K, AX, 64, SW>(exact, nt);
        if (!k) k = direct_t<K, AX, 16, SW>(exact, nt);
        return launch(k, grid, dim3(TL * ax.P), lds, with_runs(ax, grid.x, true, (AX == 1 ? 128 : 1024) / TL), cm, sw,
                      s);
    }
}

template <int AX, class SW>
int launch_t(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, hipStream_t s) {
    if constexpr (AX != 0 && SW::kFilter)
        if (ax.K == 16) return launch_k<16, AX>(ax, cm, sw, s);
    return launch_k<8, AX>(ax, cm, sw, s);
}

EulerPhys euler_phys_of(const cs_solver* sv) {
    EulerPhys ph;
    ph.umf = sv->cfg.umf;
    ph.J = sv->cfg.yaco;
    for (int a = 0; a < 3; a++) ph.m[a] = sv->cfg.metric[a];
    return ph;
}

double uf_of(const cs_solver* sv, int a) { return a == 0 ? sv->cfg.umf.x : (a == 1 ? sv->cfg.umf.y : sv->cfg.umf.z); }

// adjoint scratch: seed t and accumulator g (5 fields each), the face
// buffers mu|G of the three axes, and the tape of cs_solver_rk4_vjp
long adj_face_buf(const cs_solver* sv) { return 5 * sv->g.lmx * 2; }
long adj_tape(const cs_solver* sv) { return adj_face_buf(sv) + 2 * faces_size(sv->g); }
long adj_doubles(const cs_solver* sv) { return adj_tape(sv) + 20 * sv->g.lmx + 4 * faces_size(sv->g); }

// device table of the transposed operator `op` along the axis of t
int upload(const cs_solver* sv, int op, const AxisDesc& t, int seam, double** d) {
    std::vector<double> h, c;
    int rc = build_adjoint_table(op, t.N, seam, seam, sv->cfg.alpha_f, sv->num->pb_host, t.K, h);
    if (rc) return rc;
    chunk_table(h, t.N, t.K, t.P, c);
    CS_HIP(hipMalloc(d, c.size() * sizeof(double)));
    CS_HIP(hipMemcpy(*d, c.data(), c.size() * sizeof(double), hipMemcpyHostToDevice));
    return CS_OK;
}

// the descriptors of the transposed sweeps and the scratch.  Derivative: 8-point
// chunks: the 5 x 16 values of a 16-point one spill beside the epilogue's
// loads (128^3 y, z, carries over 48 rows: 64, 63 us against 68, 69).  Filter
// along y and z: 16-point chunks where they fit, one field a workgroup (128^3
// y, z: 32, 37 us; on 8-point chunks 54, 60 with 16 lines a workgroup).
int adjoint_setup(cs_solver* sv) {
    if (sv->adj) return CS_OK;
    int rc;
    for (int a = 0; a < 3; a++) {
        AxisDesc t = sv->ax[a], f = t;
        if (fits16(f, a)) {
            f.K = 16;
            f.P = (f.N + 15) / 16;
        }
        if (!sv->ttabs[a] && (rc = upload(sv, OP_DERIV_T, t, t.seam, &sv->ttabs[a]))) return rc;
        if (sv->cfg.filter && !f.seam && !sv->fttabs[a] && (rc = upload(sv, OP_FILTER_T, f, 0, &sv->fttabs[a])))
            return rc;
        t.tab = sv->ttabs[a];
        f.ftab = sv->fttabs[a];
        sv->tax[a] = t;
        sv->ftax[a] = f;
    }
    CS_HIP(hipMalloc(&sv->adj, sizeof(double) * adj_doubles(sv)));
    return CS_OK;
}

// transposed filter along axis a in place on the five fields of lam
template <int AX>
int filter_t_axis(cs_solver* sv, double* lam, const SweepCommon& cm, hipStream_t s) {
    const AxisDesc& ax = sv->ax[AX];
    if (ax.seam) return filter_sweeps(sv, lam, s, AX);        // cyclic: its own transpose
    const FT<AX == 0 ? 5 : 1> f{lam, sv->g.lmx, ax.ftab + 6 * ax.P * ax.K + 8};
    return launch_t<AX>(sv->ftax[AX], cm, f, s);
}

template <int AX, int MODE, bool CURV>
int stage_sweep_t(cs_solver* sv, const SweepCommon& cm, const double* q, const double* t, const double* gin,
                  double* gout, double* lam, double* tout, double ck, const double* fb, hipStream_t s) {
    const AxisDesc& ax = sv->tax[AX];
    const long lmx = sv->g.lmx;
    AT<AX, MODE, CURV> a{};
    fields(q, lmx, a.q);
    fields(t, lmx, a.t);
    fields(gin, lmx, a.gin);
    fields(gout, lmx, a.gout);
    fields(lam, lmx, a.lam);
    fields(tout, lmx, a.tout);
    if (ax.gcbc) {
        a.mu = fb + 2 * face_offset(sv->g, AX);
        a.G = a.mu + 10 * ax.nlines;
    }
    a.nface = ax.nlines;
    a.ck = ck;
    a.m = sv->cfg.metric[AX];
    a.uf = uf_of(sv, AX);
    a.umf = sv->cfg.umf;
    if constexpr (CURV) a.mt = sv->met;
    return launch_t<AX>(ax, cm, a, s);
}

// ck = dt/div times the constant Jacobian; curvilinear solvers pass a seed
// already scaled by the point's Jacobian (backward_fused) and ck = dt/div
template <int AX, int MODE>
int stage_sweep(cs_solver* sv, const SweepCommon& cm, const double* q, const double* t, const double* gin,
                double* gout, double* lam, double* tout, double ck, const double* fb, hipStream_t s) {
    if (sv->curv) return stage_sweep_t<AX, MODE, true>(sv, cm, q, t, gin, gout, lam, tout, ck, fb, s);
    // (constant Jacobian: scaling the seed or the result is the same)
    return stage_sweep_t<AX, MODE, false>(sv, cm, q, t, gin, gout, lam, tout, ck * sv->cfg.yaco, fb, s);
}

// face seeds of every non-reflective axis for the RHS evaluated at q with
// boundary derivatives `faces` ([3 axes][2][5][face]) and seed t
int face_adjoints(cs_solver* sv, const double* q, const double* t, const double* faces, const double* sbcc,
                  double* fb, hipStream_t s) {
    const EulerPhys ph = euler_phys_of(sv);
    for (int a = 0; a < 3; a++) {
        const AxisDesc& ax = sv->ax[a];
        if (!ax.gcbc) continue;
        const long nf = ax.nlines;
        double* mu = fb + 2 * face_offset(sv->g, a);
        hipLaunchKernelGGL(face_adjoint_kernel, dim3((unsigned)((2 * nf + 255) / 256)), dim3(256), 0, s, q, t, sbcc,
                           faces + face_offset(sv->g, a), mu, mu + 10 * nf, a, ax.N, nf, (long)sv->g.lxi,
                           (long)sv->g.lxi * sv->g.let, ax.st, ph, sv->g.lmx, sv->curv ? sv->met.cm[a] : nullptr,
                           sv->curv ? sv->met.J : nullptr);
        CS_HIP(hipGetLastError());
    }
    return CS_OK;
}

// out = J t, five fields: the seed of a stage's transposed RHS on a
// curvilinear grid (stage k adds -dt/div * J(x) R(q) at each point x, so its
// adjoint applies R^T to J t, the Jacobian on the output side of R)
__global__ void __launch_bounds__(256) scale_seed_kernel(const double* t, const double* J, double* out, long lmx) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= lmx) return;
    const double j = J[i];
#pragma unroll
    for (int v = 0; v < 5; v++) out[i + v * lmx] = j * t[i + v * lmx];
}

// lam <- step'(q0)^T lam from a tape (fused sweeps)
int backward_fused(cs_solver* sv, const double* tape, double* lam, double dt, const double* sbcc, hipStream_t s) {
    const long lmx = sv->g.lmx, n5 = 5 * lmx, F = faces_size(sv->g);
    const double* faces = tape + 20 * lmx;
    double* tb = sv->adj;
    double* gb = tb + n5;
    double* fb = sv->adj + adj_face_buf(sv);
    const SweepCommon cm = common_of(sv, sbcc);
    int rc;
    if (sv->cfg.filter) {
        if ((rc = filter_t_axis<2>(sv, lam, cm, s))) return rc;
        if ((rc = filter_t_axis<1>(sv, lam, cm, s))) return rc;
        if ((rc = filter_t_axis<0>(sv, lam, cm, s))) return rc;
    }
    for (int k = 4; k >= 1; k--) {
        const double* q = tape + (long)(k - 1) * n5;
        const double* t = k == 4 ? lam : tb;
        const double ck = dt / (double)(5 - k);   // times the Jacobian in stage_sweep
        if (sv->curv) {
            // the seed scaled by the point's Jacobian, in the stage buffer qc
            // (unused outside cs_solver_rk4_step)
            hipLaunchKernelGGL(scale_seed_kernel, dim3((unsigned)((lmx + 255) / 256)), dim3(256), 0, s, t, sv->met.J,
                               sv->qc, lmx);
            CS_HIP(hipGetLastError());
            t = sv->qc;
        }
        if ((rc = face_adjoints(sv, q, t, faces + (long)(k - 1) * F, sbcc, fb, s))) return rc;
        if ((rc = stage_sweep<2, 0>(sv, cm, q, t, nullptr, gb, nullptr, nullptr, 0.0, fb, s))) return rc;
        if ((rc = stage_sweep<1, 1>(sv, cm, q, t, gb, gb, nullptr, nullptr, 0.0, fb, s))) return rc;
        if (k > 1)
            rc = stage_sweep<0, 2>(sv, cm, q, t, gb, nullptr, lam, tb, ck, fb, s);
        else
            rc = stage_sweep<0, 3>(sv, cm, q, t, gb, nullptr, lam, nullptr, ck, fb, s);
        if (rc) return rc;
    }
    return CS_OK;
}

// one RK4 step in place on qa recording the tape; dt from the CFL limit when
// dt <= 0 (as cs_solver_rk4_step)
int step_recording(cs_solver* sv, double* qa, const double* sbcc, double dt, double* tape, hipStream_t s) {
    const long lmx = sv->g.lmx, n5 = 5 * lmx, F = faces_size(sv->g);
    double* faces = tape + 20 * lmx;
    int rc = time_step(sv, qa, dt, s);
    if (rc) return rc;
    CS_HIP(hipMemcpyAsync(tape, qa, sizeof(double) * n5, hipMemcpyDeviceToDevice, s));
    for (int k = 1; k <= 4 && !rc; k++) {
        sv->rec = faces + (long)(k - 1) * F;
        rc = rhs_sweeps(sv, tape + (long)(k - 1) * n5, sbcc, k < 4 ? tape + (long)k * n5 : qa, tape, 5 - k, s);
    }
    sv->rec = nullptr;
    if (rc) return rc;
    return step_filter(sv, qa, s);
}

}  // namespace

bool adjoint_fused(const cs_solver* sv) {
    if (sv->adj_mode != 1 || sv->cfg.viscous) return false;
    for (int a = 0; a < 3; a++) {
        const AxisDesc& ax = sv->ax[a];
        if (ax.K != 8 || !chunks_fit(ax.N, ax.P, 8) || ax.P > (a == 0 ? 64 : kMaxP)) return false;
    }
    return true;
}

long tape_doubles(const cs_solver* sv) { return 20 * sv->g.lmx + 4 * faces_size(sv->g); }

int rk4_step_tape(cs_solver* sv, double* qa, const double* sbcc, double dt, double* tape, hipStream_t s) {
    if (sv->cfg.viscous) return fail(CS_ERR_UNSUPPORTED, "the adjoint covers the inviscid right-hand side");
    return step_recording(sv, qa, sbcc, dt, tape, s);
}

int rk4_vjp_tape(cs_solver* sv, const double* tape, double* lam, double dt, const double* sbcc, hipStream_t s) {
    if (sv->cfg.viscous) return fail(CS_ERR_UNSUPPORTED, "the adjoint covers the inviscid right-hand side");
    if (!(dt > 0.0)) return fail(CS_ERR_ARG, "the adjoint needs the step's dt > 0");
    if (!adjoint_fused(sv)) {
        const long n5 = 5 * sv->g.lmx;
        return rk4_vjp_lines(sv, tape, tape + n5, lam, dt, sbcc, s);
    }
    int rc = adjoint_setup(sv);
    if (rc) return rc;
    return backward_fused(sv, tape, lam, dt, sbcc, s);
}

// the fused forms of cs_solver_rk4_vjp / cs_solver_rhs_vjp (adjoint_fused)
int rk4_vjp_fused(cs_solver* sv, const double* q0, double* lam, double dt, const double* sbcc, hipStream_t s) {
    int rc = adjoint_setup(sv);
    if (rc) return rc;
    const long lmx = sv->g.lmx, n5 = 5 * lmx, F = faces_size(sv->g);
    double* tape = sv->adj + adj_tape(sv);
    double* faces = tape + 20 * lmx;
    // stage states and faces of q0..q2 by the forward stages, faces of q3 by
    // one more right-hand side; dt into the device slot the stages read
    if ((rc = time_step(sv, q0, dt, s))) return rc;
    CS_HIP(hipMemcpyAsync(tape, q0, sizeof(double) * n5, hipMemcpyDeviceToDevice, s));
    for (int k = 1; k <= 4 && !rc; k++) {
        sv->rec = faces + (long)(k - 1) * F;
        if (k < 4)
            rc = rhs_sweeps(sv, tape + (long)(k - 1) * n5, sbcc, tape + (long)k * n5, tape, 5 - k, s);
        else
            rc = rhs_sweeps(sv, tape + 3 * n5, sbcc, sv->dpart, nullptr, 0, s);
    }
    sv->rec = nullptr;
    if (rc) return rc;
    return backward_fused(sv, tape, lam, dt, sbcc, s);
}

int rhs_vjp_fused(cs_solver* sv, const double* q, const double* lam, double* g, const double* sbcc, hipStream_t s) {
    int rc = adjoint_setup(sv);
    if (rc) return rc;
    double* faces = sv->adj + adj_tape(sv) + 20 * sv->g.lmx;
    double* fb = sv->adj + adj_face_buf(sv);
    sv->rec = faces;
    rc = rhs_sweeps(sv, q, sbcc, sv->dpart, nullptr, 0, s);
    sv->rec = nullptr;
    if (rc) return rc;
    const SweepCommon cm = common_of(sv, sbcc);
    if ((rc = face_adjoints(sv, q, lam, faces, sbcc, fb, s))) return rc;
    if ((rc = stage_sweep<2, 0>(sv, cm, q, lam, nullptr, g, nullptr, nullptr, 0.0, fb, s))) return rc;
    if ((rc = stage_sweep<1, 1>(sv, cm, q, lam, g, g, nullptr, nullptr, 0.0, fb, s))) return rc;
    return stage_sweep<0, 1>(sv, cm, q, lam, g, g, nullptr, nullptr, 0.0, fb, s);
}

}  // namespace fused
}  // namespace cs

extern "C" {

int cs_solver_tape_size(const cs_solver* sv, size_t* doubles) {
    if (!sv || !doubles) return cs::fail(CS_ERR_ARG, "null argument");
    *doubles = (size_t)cs::fused::tape_doubles(sv);
    return CS_OK;
}

int cs_solver_rk4_step_tape(cs_solver* sv, double* qa, const double* sbcc, double dt, double* dt_out, double* tape,
                            cs_stream stream) {
    if (!sv || !qa || !tape) return cs::fail(CS_ERR_ARG, "null argument");
    if (!sbcc && (sv->ax[0].gcbc || sv->ax[1].gcbc || sv->ax[2].gcbc))
        return cs::fail(CS_ERR_ARG, "non-reflective faces need sbcc");
    hipStream_t s = (hipStream_t)stream;
    int rc = cs::fused::rk4_step_tape(sv, qa, sbcc, dt, tape, s);
    if (rc || !dt_out) return rc;
    CS_HIP(hipMemcpyAsync(sv->dt_host, sv->dt, 3 * sizeof(double), hipMemcpyDeviceToHost, s));
    CS_HIP(hipStreamSynchronize(s));
    *dt_out = sv->dt_host[0];
    return CS_OK;
}

int cs_solver_rk4_vjp_tape(cs_solver* sv, const double* tape, double* lam, double dt, const double* sbcc,
                           cs_stream stream) {
    if (!sv || !tape || !lam) return cs::fail(CS_ERR_ARG, "null argument");
    if (!sbcc && (sv->ax[0].gcbc || sv->ax[1].gcbc || sv->ax[2].gcbc))
        return cs::fail(CS_ERR_ARG, "non-reflective faces need sbcc");
    return cs::fused::rk4_vjp_tape(sv, tape, lam, dt, sbcc, (hipStream_t)stream);
}

int cs_solver_adjoint_mode(cs_solver* sv, int mode) {
    if (!sv || (mode != 0 && mode != 1)) return cs::fail(CS_ERR_ARG, "adjoint mode is 0 or 1");
    sv->adj_mode = mode;
    return CS_OK;
}

}  // extern "C"
