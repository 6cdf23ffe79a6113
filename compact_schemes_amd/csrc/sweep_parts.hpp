// sweep_parts.hpp -- pieces shared by the line-sweep kernels of the fused
// solver (forward sweeps in fused.hip, transposed sweeps in tape.hip):
// 32-bit field offsets, line addressing, the chunked LU recurrences of the
// line solve and their carries across chunks (wave scans for x lines, LDS
// folds for y/z lines), and the host-side argument helpers.
#pragma once

#include "fused.hpp"

namespace cs {
namespace fused {

typedef unsigned int uoff;    // byte offset inside one field

__device__ __forceinline__ double ldg(const double* p, uoff bo) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(p) + bo);
}
__device__ __forceinline__ void stg(double* p, uoff bo, double v) {
    *reinterpret_cast<double*>(reinterpret_cast<char*>(p) + bo) = v;
}
// the same with the streaming hint where NT: the lines a sweep passes once and
// that no cache can hold until they are used again
template <bool NT>
__device__ __forceinline__ double ldg(const double* p, uoff bo) {
    const double* a = reinterpret_cast<const double*>(reinterpret_cast<const char*>(p) + bo);
    if constexpr (NT) return __builtin_nontemporal_load(a);
    else return *a;
}
template <bool NT>
__device__ __forceinline__ void stg(double* p, uoff bo, double v) {
    double* a = reinterpret_cast<double*>(reinterpret_cast<char*>(p) + bo);
    if constexpr (NT) __builtin_nontemporal_store(v, a);
    else *a = v;
}

struct Phys {
    cs_point umf;
    double mu, J;
    double m[3];   // metric scale per axis: xi_x, eta_y, zeta_z
};

__device__ __forceinline__ Prim prim_at(const double* const* q, uoff bo, double* qq) {
#pragma unroll
    for (int v = 0; v < 5; v++) qq[v] = ldg(q[v], bo);
    return primitive(qq);
}
// the two quantities of the time step at one point with constant diagonal
// metrics (calc_time_step_kernel, src/cuda/kernels/physics.hpp:335-427, D9
// corrected): the convective (c |grad xi| + |u . grad xi|) |J| and the
// viscous mu/rho |grad xi|^2 J^2.  One expression for every kernel that
// reduces them, so that all give the same dt bit for bit.  The viscous one is
// a product of non-negative factors rounded left to right, so its maximum
// over points is its value at the largest 1/rho (rounding is monotone).
__device__ __forceinline__ double dt_conv(const Phys& ph, double u, double v, double w, double c2) {
    const double rr1 = ph.m[0] * ph.m[0] + ph.m[1] * ph.m[1] + ph.m[2] * ph.m[2];
    const double rr2 = fabs(ph.m[0] * (u + ph.umf.x)) + fabs(ph.m[1] * (v + ph.umf.y)) +
                       fabs(ph.m[2] * (w + ph.umf.z));
    return (sqrt(c2 * rr1) + rr2) * fabs(ph.J);
}
__device__ __forceinline__ double dt_visc(const Phys& ph, double rhoi) {
    const double rr1 = ph.m[0] * ph.m[0] + ph.m[1] * ph.m[1] + ph.m[2] * ph.m[2];
    const double ssi = fabs(ph.J);
    return rhoi * ph.mu * rr1 * ssi * ssi;
}
// the same two maxima updated at one point with the point's metric rows M[a]
// = grad xi_a and Jacobian J (calc_time_step_kernel's full form); one
// expression for the separate pass and the sweep that folds it
__device__ __forceinline__ void dt_curv_point(const double (&M)[3][3], double J, const Phys& ph, const Prim& p,
                                              double& m0, double& m1) {
    const double u = p.u + ph.umf.x, v = p.v + ph.umf.y, w = p.w + ph.umf.z;
    double rr1 = 0.0, rr2 = 0.0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double mx = M[a][0], my = M[a][1], mz = M[a][2];
        rr1 += mx * mx + my * my + mz * mz;
        rr2 += fabs(mx * u + my * v + mz * w);
    }
    const double ssi = fabs(J);
    m0 = fmax(m0, (sqrt(p.c2 * rr1) + rr2) * ssi);
    m1 = fmax(m1, p.rhoi * ph.mu * rr1 * ssi * ssi);
}

// heat flux along an axis from the physical c^2 gradient and the axis's
// stress row: the last lines of viscous_closure with constant metrics, the
// same operations in the same order (with FP32 storage of the intermediates on
// the stored gradient and stress; the heat flux itself is then not rounded)
__device__ __forceinline__ double heat_flux(const Phys& ph, double c2g, double u, double v, double w, double t0,
                                            double t1, double t2) {
    const double b1 = kGamm1Prndtli * (ph.mu * ph.J);
    return b1 * c2g + u * t0 + v * t1 + w * t2;
}

// byte offset of row 0 of line f of an axis (f runs over the face's points
// with the first remaining index fastest)
__device__ __forceinline__ uoff line_off(int axis, uoff f, uoff lxi, uoff plane) {
    if (axis == 0) return f * lxi * 8u;
    if (axis == 1) return ((f / lxi) * plane + (f % lxi)) * 8u;
    return f * 8u;
}

// recurrences of the solve on the K rows of a chunk.  tab is a chunk_table:
// [6][P*K] rows nu, mu, rho, Mf, Rb, z by chunk row and 44 scalars; a padding
// row has nu = 0 and mu = rho = 1, which hands the carries on, so every chunk
// runs K rows; NP = P*K.  The products that are fused are named, so that every
// kernel rounds alike.
template <int K, int NF>
__device__ __forceinline__ void forward_local(const double* tab, int NP, int s, double (&r)[NF][K],
                                              double (&carry)[NF]) {
#pragma unroll
    for (int f = 0; f < NF; f++) carry[f] = 0.0;
#pragma unroll
    for (int t = 0; t < K; t++) {
        const double nu = tab[s + t], mu = tab[NP + s + t];
#pragma unroll
        for (int f = 0; f < NF; f++) {
            carry[f] = __builtin_fma(nu, r[f][t], mu * carry[f]);
            r[f][t] = carry[f];
        }
    }
}

template <int K, int NF>
__device__ __forceinline__ void backward_local(const double* tab, int NP, int s, double (&r)[NF][K],
                                               double (&carry)[NF]) {
#pragma unroll
    for (int f = 0; f < NF; f++) carry[f] = 0.0;
#pragma unroll
    for (int t = K - 1; t >= 0; t--) {
        const double rh = tab[2 * NP + s + t];
#pragma unroll
        for (int f = 0; f < NF; f++) {
            carry[f] = __builtin_fma(rh, carry[f], r[f][t]);
            r[f][t] = carry[f];
        }
    }
}

template <int K, int NF>
__device__ __forceinline__ void apply_carry(const double* tab, int off, int s, double (&r)[NF][K],
                                            const double (&G)[NF]) {
#pragma unroll
    for (int t = 0; t < K; t++) {
        const double M = tab[off + s + t];
#pragma unroll
        for (int f = 0; f < NF; f++) r[f][t] = __builtin_fma(M, G[f], r[f][t]);
    }
}

// Every chunk of a line counts in a carry: a row reaches every other of its
// line, by a factor of (3 - sqrt 5)/2 = 0.382 a row along a derivative, 0.82
// along a filter at alpha_f = 0.49, and a NaN or an infinity whole.  Folding a
// derivative's carries over the nearest 48 rows alone loses that for 1.6 % of
// a step at 256^3 (10.27 against 10.11 ms) and 2.9 % at 150x133x97 (1.72
// against 1.67).  kCarryRows is the longest line of the sweep kernels.
constexpr int kCarryRows = 1024;

// carries across the chunks of a line through LDS: buf = [NF][P][TL].  One field
// folds two chunks an iteration: left to itself the compiler unrolls further,
// code that the smallest launches wait for (six operators on 64^3 33.2 against
// 32.2 us, sixteen blocks batched 2577 against 2525); four or five fields by
// two are slower (512x288x96 step 8322 -> 8404).
template <int NF, int K>
__device__ __forceinline__ void fold_forward(const double* buf, const double* tab, int NP, int P, int TL, int c,
                                             int lloc, double (&G)[NF]) {
#pragma unroll
    for (int f = 0; f < NF; f++) G[f] = 0.0;
    auto step = [&](int cc) {
        const double M = tab[3 * NP + cc * K + K - 1];
#pragma unroll
        for (int f = 0; f < NF; f++) G[f] = __builtin_fma(M, G[f], buf[(f * P + cc) * TL + lloc]);
    };
    if constexpr (NF == 1) {
#pragma unroll 2
        for (int cc = 0; cc < c; cc++) step(cc);
    } else {
        for (int cc = 0; cc < c; cc++) step(cc);
    }
}

template <int NF, int K>
__device__ __forceinline__ void fold_backward(const double* buf, const double* tab, int NP, int P, int TL, int c,
                                              int lloc, double (&X)[NF]) {
#pragma unroll
    for (int f = 0; f < NF; f++) X[f] = 0.0;
    auto step = [&](int cc) {
        const double R = tab[4 * NP + cc * K];
#pragma unroll
        for (int f = 0; f < NF; f++) X[f] = __builtin_fma(R, X[f], buf[(f * P + cc) * TL + lloc]);
    };
    if constexpr (NF == 1) {
#pragma unroll 2
        for (int cc = P - 1; cc > c; cc--) step(cc);
    } else {
        for (int cc = P - 1; cc > c; cc--) step(cc);
    }
}

// carries across the chunks of a line held by P consecutive lanes of a wave
// (c = lane's chunk): segmented Kogge-Stone scans of the affine maps
// x -> A*x + B
template <int NF>
__device__ __forceinline__ void scan_forward(double A, const double (&carry)[NF], int c, int P, double (&G)[NF]) {
    double B[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) B[f] = carry[f];
    for (int d = 1; d < P; d <<= 1) {
        const double Au = __shfl_up(A, d);
        double Bu[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) Bu[f] = __shfl_up(B[f], d);
        if (c >= d) {
#pragma unroll
            for (int f = 0; f < NF; f++) B[f] = __builtin_fma(A, Bu[f], B[f]);
            A *= Au;
        }
    }
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const double g = __shfl_up(B[f], 1);
        G[f] = (c == 0) ? 0.0 : g;
    }
}

template <int NF>
__device__ __forceinline__ void scan_backward(double A, const double (&carry)[NF], int c, int P, double (&X)[NF]) {
    double B[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) B[f] = carry[f];
    for (int d = 1; d < P; d <<= 1) {
        const double Ad = __shfl_down(A, d);
        double Bd[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) Bd[f] = __shfl_down(B[f], d);
        if (c + d < P) {
#pragma unroll
            for (int f = 0; f < NF; f++) B[f] = __builtin_fma(A, Bd[f], B[f]);
            A *= Ad;
        }
    }
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const double x = __shfl_down(B[f], 1);
        X[f] = (c + 1 < P) ? x : 0.0;
    }
}

// workgroup -> line group.  Workgroups are dispatched round-robin over the 8
// XCDs, each with its own L2; xcd = 1 + log2(G) gives runs of G neighbouring
// groups to one XCD (0: plain order).
__device__ __forceinline__ long group_of(int xcd) {
    const unsigned w = blockIdx.x;
    if (!xcd) return w;
    const int g = xcd - 1;
    const unsigned span = 8u << g, i = w / 8;
    if (w >= gridDim.x / span * span) return w;
    return (i >> g) * span + ((w % 8) << g) + (i & ((1u << g) - 1));
}

// LDS slot of row t of chunk c of line li in the transposing x kernels
template <int K>
__device__ __forceinline__ int xt_slot(int li, int P, int c, int t) { return (li * P + c) * (K + 1) + t; }

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
inline Phys phys_of(const cs_solver* sv) {
    Phys ph;
    ph.umf = sv->cfg.umf;
    ph.mu = sv->cfg.mu;
    ph.J = sv->cfg.yaco;
    for (int a = 0; a < 3; a++) ph.m[a] = sv->cfg.metric[a];
    return ph;
}

inline SweepCommon common_of(const cs_solver* sv, const double* sbcc) {
    SweepCommon cm;
    cm.lxi = sv->g.lxi;
    cm.plane = (long)sv->g.lxi * sv->g.let;
    cm.pb = sv->num->pb;
    cm.sbcc = sbcc;
    return cm;
}

// offset of axis a's [2 face][5 var][face] block in a buffer holding the
// three axes' boundary-derivative faces, and that buffer's size
inline long face_offset(const Geo& g, int a) {
    long o = 0;
    for (int b = 0; b < a; b++) o += 10 * g.face_size(b);
    return o;
}
inline long faces_size(const Geo& g) { return face_offset(g, 3); }

template <class T, int N>
inline void fields(T* base, long lmx, T* (&out)[N]) {
    for (int k = 0; k < N; k++) out[k] = base ? base + (long)k * lmx : nullptr;
}

}  // namespace fused
}  // namespace cs
