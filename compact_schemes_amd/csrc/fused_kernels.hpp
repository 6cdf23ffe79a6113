// fused_kernels.hpp -- the sweep functors, kernels and launchers of the
// fused right-hand side (see fused.hip for the design), shared by the
// translation units that instantiate them: fused.hip (FP64 intermediates) and
// fused_f32.hip (the viscous intermediates stored in FP32).
#pragma once

#include <type_traits>

#include "sweep_parts.hpp"

namespace cs {
namespace fused {

// loads and stores of a field of storage type TS at the byte offset of the
// point in an FP64 field (an FP32 field holds the same points at half the offset)
template <bool NT>
__device__ __forceinline__ double ldr(const double* p, uoff bo) { return ldg<NT>(p, bo); }
template <bool NT>
__device__ __forceinline__ float ldr(const float* p, uoff bo) {
    const float* a = reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + (bo >> 1));
    if constexpr (NT) return __builtin_nontemporal_load(a);
    else return *a;
}
template <bool NT>
__device__ __forceinline__ void stv(double* p, uoff bo, double v) { stg<NT>(p, bo, v); }
template <bool NT>
__device__ __forceinline__ void stv(float* p, uoff bo, double v) {
    float* a = reinterpret_cast<float*>(reinterpret_cast<char*>(p) + (bo >> 1));
    if constexpr (NT) __builtin_nontemporal_store((float)v, a);
    else *a = (float)v;
}

// a sweep's values at one point
template <bool NT, class SW>
__device__ __forceinline__ void point(const SW& sw, uoff bo, double* v) {
    typename SW::Raw w;
    sw.template load<NT>(bo, w);
    sw.eval(w, v);
}

template <bool NT, class SW>
__device__ __forceinline__ void add_out(const SW& sw, uoff bo, double* d) {
    if constexpr (SW::kAdds) {
        typename SW::Out e;
        sw.template load_out<NT>(bo, e);
        sw.add_out(e, d);
    }
}

// ---------------------------------------------------------------------------
// sweep functors
// ---------------------------------------------------------------------------
// S1: velocity and c^2 gradients along AX.  The first two S1 sweeps of an
// RHS store their index-space gradients; the third (CLOSE) combines its own
// gradients with the stored ones into the stress tensor and the heat flux.
// With constant metrics the heat flux along an axis needs the c^2 gradient
// along that axis alone, so CLOSE forms its own component and the flux sweeps
// of the other two axes form theirs from the stored gradient (S2T): 32 bytes a
// point less (256^3 S1x 526 -> 430 us).
template <int AX, bool CLOSE, class TS, bool CURV = false, bool DT = false>
struct S1T {
    typedef TS Store;                      // storage type of the gradients, stress and heat flux
    static constexpr bool kCurv = CURV;    // per-point metrics (curvilinear solvers)
    static constexpr int NF = 4;
    static constexpr bool kGcbc = false;   // gradients only; BC updates act on the flux sweeps
    static constexpr bool kBlocks = false;
    // memory the sweep takes per point (streaming rule of the launch)
    static constexpr int kBytes = 40 + (int)sizeof(TS) * (CLOSE ? (CURV ? 17 : 13) : 4) + (CURV && CLOSE ? 80 : 0);
    // the transposing x kernel keeps u, v, w of its points in LDS for the
    // closure (store_pv) instead of reading q again
    static constexpr int kStash = CLOSE ? 3 : 0;
    static constexpr int kH = 2;           // derivative stencil half-width
    static constexpr int kWpe = 3;         // waves per SIMD of the y/z kernels (168 VGPRs)
    static constexpr int kWpe16 = 2;       // with 16-point chunks
    static constexpr bool kEnds = false;   // end_value takes the results at a line's ends
    static constexpr bool kFilter = false;
    // DT: a sweep that also reduces the time step's maxima over the points it
    // evaluates, one pair per workgroup: a y/z gradient sweep
    // (constant metrics), or the closing x sweep with per-point metrics, which
    // loads the metric rows and J of every point anyway
    static constexpr bool kDt = DT;
    static_assert(!DT || (!CLOSE && !CURV && AX != 0) || (CLOSE && CURV && AX == 0),
                  "time-step maxima: y/z gradient sweeps of constant metrics, closing x sweep of per-point metrics");
    const double* q[5];
    TS* gout[4];              // !CLOSE: d/d(axis AX) of u, v, w, c^2
    const TS* gin[3][4];      // CLOSE: stored gradients along the other two axes
    TS* tau[6];               // xx, yy, zz, xy, yz, zx
    TS* hf[3];                // CURV: all, else component AX
    Phys ph;
    Metric mt;                // CURV: the point's metric rows and Jacobian
    double* dtpart;           // kDt: the workgroup's two time-step maxima [2*blockIdx.x]

    // a point's inputs, and its values from them (two steps, so that a kernel
    // can have the loads of several points in flight)
    struct Raw { double q[5]; };
    template <bool NT>
    __device__ __forceinline__ void load(uoff bo, Raw& w) const {
#pragma unroll
        for (int v = 0; v < 5; v++) w.q[v] = ldg<NT>(q[v], bo);
    }
    __device__ __forceinline__ void eval(const Raw& w, double* v) const {
        const Prim p = primitive(w.q);
        v[0] = p.u;
        v[1] = p.v;
        v[2] = p.w;
        v[3] = p.c2;
    }
    // eval() and the largest 1/rho so far (kDt)
    __device__ __forceinline__ void eval_dt(const Raw& w, double* v, double& rhoi_max) const {
        const Prim p = primitive(w.q);
        v[0] = p.u;
        v[1] = p.v;
        v[2] = p.w;
        v[3] = p.c2;
        rhoi_max = fmax(rhoi_max, p.rhoi);
    }
    static constexpr bool kAdds = false;
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d) const {
        if constexpr (!CLOSE) {
#pragma unroll
            for (int f = 0; f < 4; f++) stv<NT>(gout[f], bo, d[f]);
        } else {
            double qq[5];
            const Prim p = prim_at(q, bo, qq);      // q of this point: just read by this sweep
            const double uvw[3] = {p.u, p.v, p.w};
            close<NT>(bo, d, uvw);
        }
    }
    // the store of the closing sweep with u, v, w of the point supplied
    template <bool NT>
    __device__ __forceinline__ void store_pv(uoff bo, const double* d, const double* uvw) const {
        if constexpr (CLOSE) close<NT>(bo, d, uvw);
        else store<NT>(bo, d);
    }
    // the same, updating the time step's maxima mm[0..1] at the point (kDt, CURV)
    template <bool NT>
    __device__ __forceinline__ void store_pv_dt(uoff bo, const double* d, const double* uvw, double* mm) const {
        close_dt<NT, true>(bo, d, uvw, mm);
    }
    template <bool NT>
    __device__ __forceinline__ void close(uoff bo, const double* d, const double* uvw) const {
        close_dt<NT, false>(bo, d, uvw, nullptr);
    }
    template <bool NT, bool WITH_DT>
    __device__ __forceinline__ void close_dt(uoff bo, const double* d, const double* uvw, double* mm) const {
        double gr[3][4];
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int f = 0; f < 4; f++)
                gr[a][f] = (a == AX) ? d[f] : (f < 3 || CURV) ? (double)ldr<NT>(gin[a][f], bo) : 0.0;
        // chain rule of calc_viscous_shear_stress_post_compute_kernel
        // (src/cuda/kernels/physics.hpp:267-281): d/dx_k = sum_a m_a[k] d/dxi_a
        double g[9], c2g[3], J = ph.J;
        double M[3][3];
        if constexpr (CURV) {
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
                for (int k = 0; k < 3; k++) M[a][k] = ldg<NT>(mt.m[a][k], bo);
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < 3; k++) g[3 * f + k] = M[0][k] * gr[0][f] + M[1][k] * gr[1][f] + M[2][k] * gr[2][f];
#pragma unroll
            for (int k = 0; k < 3; k++) c2g[k] = M[0][k] * gr[0][3] + M[1][k] * gr[1][3] + M[2][k] * gr[2][3];
            J = ldg<NT>(mt.J, bo);
        } else {
            // diagonal metrics: m_a[k] = m[a] for k = a
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int a = 0; a < 3; a++) g[3 * f + a] = ph.m[a] * gr[a][f];
#pragma unroll
            for (int a = 0; a < 3; a++) c2g[a] = ph.m[a] * gr[a][3];
        }
        double t6[6], h3[3], d4;
        viscous_closure(ph.mu, J, g, c2g, uvw, t6, h3, &d4);
#pragma unroll
        for (int k = 0; k < 6; k++) stv<NT>(tau[k], bo, t6[k]);
#pragma unroll
        for (int k = 0; k < 3; k++)
            if (CURV || k == AX) stv<NT>(hf[k], bo, h3[k]);
        if constexpr (WITH_DT && CURV) {
            // the point's q again (this sweep read it for the gradients)
            double qq[5];
            dt_curv_point(M, J, ph, prim_at(q, bo, qq), mm[0], mm[1]);
        }
    }
};

// the gradient sweeps with FP64 intermediates, and with FP32 ones
// (cs_solver_set_precision 1); the names the kernels carry
template <int AX, bool CLOSE>
struct S1 : S1T<AX, CLOSE, double> {};
template <int AX, bool CLOSE>
struct S1F : S1T<AX, CLOSE, float> {};
// curvilinear solvers (cs_solver_set_metrics): FP64 intermediates
template <int AX, bool CLOSE>
struct S1C : S1T<AX, CLOSE, double, true> {};
template <int AX, bool CLOSE>
struct S1CF : S1T<AX, CLOSE, float, true> {};
// the first gradient sweep of an RK4 step, reducing the time step as well
template <int AX, bool CLOSE>
struct S1D : S1T<AX, CLOSE, double, false, true> {};
template <int AX, bool CLOSE>
struct S1FD : S1T<AX, CLOSE, float, false, true> {};
// the closing sweep of an RK4 step's first stage with per-point metrics,
// reducing the time step as well
template <int AX, bool CLOSE>
struct S1CD : S1T<AX, CLOSE, double, true, true> {};
template <int AX, bool CLOSE>
struct S1CFD : S1T<AX, CLOSE, float, true, true> {};

// S2: flux divergence along AX.  MODE 0: write the partial RHS; 1: add to it;
// 2: add and write the RHS; 3: add and write q0 - dtk*J*RHS (RK stage).
template <int AX, int MODE, bool VISC, class TS, bool CURV = false>
struct S2T {
    typedef TS Store;
    static constexpr bool kCurv = CURV;    // per-point metrics (curvilinear solvers)
    static constexpr int NF = 5;
    static constexpr bool kGcbc = true;
    static constexpr bool kBlocks = CURV;
    static constexpr int kBytes = 80 + (VISC ? (int)sizeof(TS) * (CURV ? 9 : 4) : 0) + (CURV ? 24 : 0) +
                                  (MODE == 2 ? 40 : MODE == 3 ? 80 : 0);
    static constexpr int kStash = 0;
    static constexpr int kH = 2;
    static constexpr int kWpe = 3;
    static constexpr int kWpe16 = 2;
    static constexpr bool kEnds = false;
    static constexpr bool kFilter = false;
    const double* q[5];
    const TS* tr[3];          // row AX of the stress tensor
    // constant metrics: heat flux component AX in the last sweep (MODE 2, 3:
    // the closing axis), else the c^2 gradient along AX it is formed from
    static constexpr bool kHeat = VISC && !CURV && MODE < 2;
    const TS* hx;
    const TS* tau6[6];        // CURV: the whole stress tensor (xx, yy, zz, xy, yz, zx)
    const TS* h3[3];          // CURV: the whole heat flux
    Metric mt;                // CURV: the point's metric rows, Jacobian, face normals
    const double* din[5];
    double* dout[5];
    const double* q0[5];
    const double* dtp;
    int div;
    Phys ph;
    double* rec;              // [2 face][5 var][face] boundary derivatives of this sweep, or null
    long nface;
    int lxi;
    long plane;

    // the inputs of the flux at a point: the state; with VISC the stress row
    // and heat flux component of the sweep (CURV: all of them), the point's
    // metric row.  The sweep with the stage update keeps q in the caches: in
    // the first stage its q0 is the same array.
    struct Raw {
        double q[5];
        TS t[VISC ? (CURV ? 9 : 4) : 1];
        double m[CURV ? 3 : 1];
    };
    template <bool NT>
    __device__ __forceinline__ void load(uoff bo, Raw& w) const {
#pragma unroll
        for (int v = 0; v < 5; v++) w.q[v] = ldg<NT && MODE != 3>(q[v], bo);
        if constexpr (CURV) {
#pragma unroll
            for (int k = 0; k < 3; k++) w.m[k] = ldg<NT>(mt.m[AX][k], bo);
        }
        if constexpr (VISC && CURV) {
#pragma unroll
            for (int k = 0; k < 6; k++) w.t[k] = ldr<NT>(tau6[k], bo);
#pragma unroll
            for (int k = 0; k < 3; k++) w.t[6 + k] = ldr<NT>(h3[k], bo);
        } else if constexpr (VISC) {
#pragma unroll
            for (int k = 0; k < 3; k++) w.t[k] = ldr<NT>(tr[k], bo);
            w.t[3] = ldr<NT>(hx, bo);
        }
    }
    // the AX row of calc_fluxes_pre_compute_kernel with metric row m*e_AX
    // (src/cuda/kernels/physics.hpp:98-191); zero metric terms dropped
    __device__ __forceinline__ void eval(const Raw& w, double* F) const {
        const double* qq = w.q;
        const Prim p = primitive(qq);
        if constexpr (CURV) {
            // the AX row with the point's metric row (m0, m1, m2)
            const double m0 = w.m[0], m1 = w.m[1], m2 = w.m[2];
            const double ss = m0 * (p.u + ph.umf.x) + m1 * (p.v + ph.umf.y) + m2 * (p.w + ph.umf.z);
            F[0] = qq[0] * ss;
            F[1] = qq[1] * ss + m0 * p.p;
            F[2] = qq[2] * ss + m1 * p.p;
            F[3] = qq[3] * ss + m2 * p.p;
            F[4] = (qq[4] + p.p) * ss - p.p * (ph.umf.x * m0 + ph.umf.y * m1 + ph.umf.z * m2);
            if constexpr (VISC) {
                const double txx = w.t[0], tyy = w.t[1], tzz = w.t[2], txy = w.t[3], tyz = w.t[4], tzx = w.t[5];
                F[1] -= m0 * txx + m1 * txy + m2 * tzx;
                F[2] -= m0 * txy + m1 * tyy + m2 * tyz;
                F[3] -= m0 * tzx + m1 * tyz + m2 * tzz;
                F[4] -= m0 * (double)w.t[6] + m1 * (double)w.t[7] + m2 * (double)w.t[8];
            }
        } else {
            const double m = ph.m[AX];
            const double vel = (AX == 0) ? p.u : (AX == 1 ? p.v : p.w);
            const double uf = (AX == 0) ? ph.umf.x : (AX == 1 ? ph.umf.y : ph.umf.z);
            const double ss = m * (vel + uf);
            F[0] = qq[0] * ss;
            F[1] = qq[1] * ss;
            F[2] = qq[2] * ss;
            F[3] = qq[3] * ss;
            F[1 + AX] += m * p.p;
            F[4] = (qq[4] + p.p) * ss - p.p * (uf * m);
            if constexpr (VISC) {
                F[1] -= m * (double)w.t[0];
                F[2] -= m * (double)w.t[1];
                F[3] -= m * (double)w.t[2];
                double h = w.t[3];
                if constexpr (kHeat) h = heat_flux(ph, m * h, p.u, p.v, p.w, w.t[0], w.t[1], w.t[2]);
                F[4] -= m * h;
            }
        }
    }
    // the epilogue: what the sweep adds to at a point (the partial sum; with
    // the stage update also q0 and the Jacobian), and its result from that.
    // The kernels load before their first store: dout may alias din or q0 for
    // all the compiler knows, so a load placed after a store waits for it, and
    // interleaved they would run one memory round trip per field and row.
    static constexpr bool kAdds = MODE != 0;
    struct Out {
        double din[5], q0[MODE == 3 ? 5 : 1], J;
    };
    template <bool NT>
    __device__ __forceinline__ void load_out(uoff bo, Out& e) const {
#pragma unroll
        for (int f = 0; f < 5; f++) e.din[f] = ldg<NT>(din[f], bo);
        if constexpr (MODE == 3) {
#pragma unroll
            for (int f = 0; f < 5; f++) e.q0[f] = ldg(q0[f], bo);
            e.J = CURV ? ldg<NT>(mt.J, bo) : ph.J;
        }
    }
    __device__ __forceinline__ void add_out(const Out& e, double* d) const {
        if constexpr (MODE == 3) {
            const double fj = dtp[0] / (double)div * e.J;
#pragma unroll
            for (int f = 0; f < 5; f++) {
                const double de = e.din[f] + d[f];
                d[f] = e.q0[f] - fj * de;
            }
        } else {
#pragma unroll
            for (int f = 0; f < 5; f++) d[f] = e.din[f] + d[f];
        }
    }
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d) const {
#pragma unroll
        for (int f = 0; f < 5; f++) stg<NT>(dout[f], bo, d[f]);
    }
    // what the characteristic BC reads at a face point: the state, the weight
    // and (curvilinear solvers) the caller's face normal and the Jacobian
    struct FaceIn {
        double q[5], w, cm[3], J;
        long fi;          // face index (x: k*let+j, y: k*lxi+i, z: j*lxi+i)
    };
    __device__ __forceinline__ FaceIn face_in(uoff bo, int face, const double* sbcc) const {
        FaceIn in;
        const long o = bo / 8u;
        in.fi = AX == 0 ? o / lxi : (AX == 1 ? (o / plane) * lxi + o % lxi : o % plane);
#pragma unroll
        for (int v = 0; v < 5; v++) in.q[v] = ldg(q[v], bo);
        in.w = ldg(sbcc, bo);
        if constexpr (CURV) {
            // [2 face][3][face], as gcbc_go takes them
            const double* c = mt.cm[AX] + (long)face * 3 * nface + in.fi;
            in.cm[0] = c[0];
            in.cm[1] = c[nface];
            in.cm[2] = c[2 * nface];
            in.J = ldg(mt.J, bo);
        } else {
            // unit normal of the face: grad(xi_AX) / |grad(xi_AX)|, grad(xi_AX) = J * metric * e_AX
            const double sg = ph.m[AX] * ph.J < 0.0 ? -1.0 : 1.0;
            in.cm[0] = AX == 0 ? sg : 0.0;
            in.cm[1] = AX == 1 ? sg : 0.0;
            in.cm[2] = AX == 2 ? sg : 0.0;
            in.J = ph.J;
        }
        return in;
    }
    // non-reflective characteristic correction at a face point from the
    // boundary derivatives of this sweep (gcbc_setup_kernel +
    // gcbc_update_non_reflective_kernel, src/cuda/kernels/gcbc.hpp:251-454)
    __device__ __forceinline__ void gcbc(const FaceIn& in, int face, const double* drv, double* corr) const {
        if (rec) {
#pragma unroll
            for (int v = 0; v < 5; v++) rec[(face * 5 + v) * nface + in.fi] = drv[v];
        }
        const Prim p = primitive(in.q);
        const double J = in.J;
        const double* cm = in.cm;
        Eig e;
        e.eleme(cm, in.q[0], in.q + 1, p.p, ph.umf);
        double cha[5], ch[5];
#pragma unroll
        for (int v = 0; v < 5; v++) cha[v] = J * drv[v];
        e.l_apply(cm, cha, ch);
        const double ra0 = 1 - 2 * face;
        double dl[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (ra0 * (e.vn + e.vs + e.ao) > 0) dl[3] = -ch[3];
        if (ra0 * (e.vn + e.vs - e.ao) > 0) dl[4] = -ch[4];
        e.r_apply(cm, dl, corr);
        // D25: a change of J*de (the amplitudes were formed from J*drv), so de changes by corr / J
#pragma unroll
        for (int v = 0; v < 5; v++) corr[v] /= J;
    }
};

template <int AX, int MODE, bool VISC>
struct S2 : S2T<AX, MODE, VISC, double> {};
template <int AX, int MODE, bool VISC>
struct S2F : S2T<AX, MODE, VISC, float> {};
template <int AX, int MODE, bool VISC>
struct S2C : S2T<AX, MODE, VISC, double, true> {};
template <int AX, int MODE, bool VISC>
struct S2CF : S2T<AX, MODE, VISC, float, true> {};

// SF: the compact filter of the five conserved variables along AX, in place
// (the filter of cs_filter: 10th-order interior rows, reduced-order centred
// rows with graded alpha near closure ends, identity end rows; cyclic on seam
// axes)
template <int AX>
struct SF {
    static constexpr int NF = 5;
    static constexpr bool kBlocks = false;
    static constexpr int kBytes = 40;
    static constexpr bool kGcbc = false;
    static constexpr int kStash = 0;
    static constexpr int kH = 5;
    static constexpr int kWpe = 3;
    static constexpr int kWpe16 = 2;
    static constexpr bool kEnds = false;
    static constexpr bool kFilter = true;
    double* q[5];
    struct Raw { double q[5]; };
    template <bool NT>
    __device__ __forceinline__ void load(uoff bo, Raw& w) const {
#pragma unroll
        for (int f = 0; f < 5; f++) w.q[f] = ldg<NT>(q[f], bo);
    }
    __device__ __forceinline__ void eval(const Raw& w, double* v) const {
#pragma unroll
        for (int f = 0; f < 5; f++) v[f] = w.q[f];
    }
    static constexpr bool kAdds = false;
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d) const {
#pragma unroll
        for (int f = 0; f < 5; f++) stg<NT>(q[f], bo, d[f]);
    }
};

// SF1: the same filter, one conserved variable per workgroup (blockIdx.y picks
// the variable of the five stored lmx points apart); a fifth of SF's registers
template <int AX>
struct SF1 {
    static constexpr int NF = 1;
    static constexpr bool kBlocks = false;
    static constexpr int kBytes = 8;
    static constexpr bool kGcbc = false;
    static constexpr int kStash = 0;
    static constexpr int kH = 5;
    static constexpr int kWpe = 3;
    static constexpr int kWpe16 = 2;
    static constexpr bool kEnds = false;
    static constexpr bool kFilter = true;
    double* q;
    long lmx;
    __device__ __forceinline__ double* field() const { return q + (long)blockIdx.y * lmx; }
    struct Raw { double q; };
    template <bool NT>
    __device__ __forceinline__ void load(uoff bo, Raw& w) const { w.q = ldg<NT>(field(), bo); }
    __device__ __forceinline__ void eval(const Raw& w, double* v) const { v[0] = w.q; }
    static constexpr bool kAdds = false;
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d) const { stg<NT>(field(), bo, d[0]); }
};

// ---------------------------------------------------------------------------
// pieces shared by the sweep kernels
//
// A line of N rows is cut into P = ceil(N/K) chunks of K rows.  Where N is
// not P*K, the D = P*K - N chunks after the first hold K-1 rows (Chunks), so
// that the first and the last chunk, with the closure, seam and face rows,
// are always whole and only the halo exchange has to look at a chunk's
// length.  The missing row is a padding row at the chunk's end whose table
// entries pass the recurrences through (chunk_table).
// ---------------------------------------------------------------------------
template <int K, bool EX>
struct Chunks {
    int D;
    __device__ __forceinline__ Chunks(int N, int P) : D(EX ? 0 : P * K - N) {}
    __device__ __forceinline__ int start(int c) const { return EX ? c * K : c * K - min(max(c - 1, 0), D); }
    __device__ __forceinline__ bool whole(int c) const { return EX || c == 0 || c > D; }
};

// rows K-H..K-1 of the window's own part and the H halo rows after it: a
// chunk of K-1 rows has its halo one row earlier
template <int K, int H, int W>
__device__ __forceinline__ void close_window(double (&w)[W], const double (&right)[H], bool whole) {
#pragma unroll
    for (int k = 0; k < H; k++) w[K + H + k] = whole ? right[k] : (k + 1 < H ? right[k + 1 < H ? k + 1 : 0] : 0.0);
    w[K + H - 1] = whole ? w[K + H - 1] : right[0];
}

// interior rows and closure rows from a window w[u] holding rows s-2+u
// (build_system, numerics_device_pc.hpp:176-293)
template <int K, int W>
__device__ __forceinline__ void window_rhs(const double (&w)[W], double (&r)[K], bool first, bool last) {
#pragma unroll
    for (int t = 0; t < K; t++) r[t] = kAa * (w[t + 3] - w[t + 1]) + kBb * (w[t + 4] - w[t]);
    if (first) {
        r[0] = kAb00 * w[2] + kAb01 * w[3] + kAb02 * w[4];
        r[1] = kAb10 * (w[4] - w[2]);
    }
    if (last) {
        r[K - 1] = -(kAb00 * w[K + 1] + kAb01 * w[K] + kAb02 * w[K - 1]);
        r[K - 2] = -kAb10 * (w[K - 1] - w[K + 1]);
    }
}

// filter rows from a window w[u] holding rows s-5+u: 10th order inside,
// order 2*dist at distance dist < 5 from a closure end, identity at the end
// (an = the order-2M coefficient sets, an[6M..6M+M], each for its row's
// alpha; the alphas enter through the LU tables); cyclic lines are all
// inside rows
template <int K, int W>
__device__ __forceinline__ void filter_rhs(const double (&w)[W], double (&r)[K], bool first, bool last,
                                           const double* an) {
    constexpr int H = 5;
#pragma unroll
    for (int t = 0; t < K; t++) {
        double v = an[30] * w[t + H];
#pragma unroll
        for (int m = 1; m <= 5; m++) v = __builtin_fma(0.5 * an[30 + m], w[t + H + m] + w[t + H - m], v);
        r[t] = v;
    }
#pragma unroll
    for (int end = 0; end < 2; end++) {
        if (end == 0 ? first : last) {
#pragma unroll
            for (int dist = 0; dist < H; dist++) {
                const int t = end == 0 ? dist : K - 1 - dist;
                double v = w[t + H];
                if (dist > 0) {
                    v = an[6 * dist] * w[t + H];
#pragma unroll
                    for (int m = 1; m <= dist; m++)
                        v = __builtin_fma(0.5 * an[6 * dist + m], w[t + H + m] + w[t + H - m], v);
                }
                r[t] = v;
            }
        }
    }
}

// Sherman-Morrison correction of a cyclic filter solve: y0 and yN1 are the
// solution of the modified system at rows 0 and N-1 (tab layout of
// chunk_table: z at 5NP, 1/(1 + z0 + kappa zN1) at 6NP, kappa at 6NP+1)
template <int K, int NF>
__device__ __forceinline__ void cyclic_correction(const double* tab, int NP, int s, const double (&y0)[NF],
                                                  const double (&yN1)[NF], double (&r)[NF][K]) {
    const double* z = tab + 5 * NP;
    const double inv = tab[6 * NP], kappa = tab[6 * NP + 1];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const double beta = (y0[f] + kappa * yN1[f]) * inv;
#pragma unroll
        for (int t = 0; t < K; t++) r[f][t] -= beta * z[s + t];
    }
}

// the same rows as window_rhs for rows s..s+L-1 of a chunk, streamed through
// a 5-row register window so that only the rows a right-hand side needs are
// live (rows from an LDS tile); zero in the padding rows
template <int K, int NF, class ROW>
__device__ __forceinline__ void stream_rhs(ROW&& row_of, double (&r)[NF][K], int s, int L, int N, bool seam) {
    constexpr int W = K + 4;
    double w0[NF], w1[NF], w2[NF], w3[NF], w4[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) w0[f] = w1[f] = w2[f] = w3[f] = w4[f] = 0.0;
#pragma unroll
    for (int u = 0; u < W; u++) {
        double v[NF];
        row_of(u, v);
#pragma unroll
        for (int f = 0; f < NF; f++) { w0[f] = w1[f]; w1[f] = w2[f]; w2[f] = w3[f]; w3[f] = w4[f]; w4[f] = v[f]; }
        if (u >= 4) {
            const int t = u - 4, j = s + t;
#pragma unroll
            for (int f = 0; f < NF; f++) {
                double x = kAa * (w3[f] - w1[f]) + kBb * (w4[f] - w0[f]);
                if (!seam) {
                    if (t == 0 && j == 0) x = kAb00 * w2[f] + kAb01 * w3[f] + kAb02 * w4[f];
                    if (t == 1 && j == 1) x = kAb10 * (w3[f] - w1[f]);
                    if (j == N - 2) x = -kAb10 * (w1[f] - w3[f]);
                    if (j == N - 1) x = -(kAb00 * w2[f] + kAb01 * w1[f] + kAb02 * w0[f]);
                }
                r[f][t] = t < L ? x : 0.0;
            }
        }
    }
}

// zero in the padding row of a chunk of K-1 rows, before the backward recurrence
template <int K, int NF>
__device__ __forceinline__ void zero_padding(double (&r)[NF][K], bool whole) {
#pragma unroll
    for (int f = 0; f < NF; f++) r[f][K - 1] = whole ? r[f][K - 1] : 0.0;
}

// quasi-disjoint seam rows, wrapped onto the opposite end of the line
// (build_system seam branch, numerics_device_pc.hpp:199-282, with the
// neighbour sums formed as fill_gpu_buffer_kernel does, kernels/numerics_pc.hpp:86-121).
// For the chunk at the line's start (end = 0) or end (end = 1; L rows):
// row(e, i, v) gives the values at distance i from end e.
template <int K, int NF, class ROW>
__device__ __forceinline__ void seam_rows(ROW&& row, int end, int L, const double* pb, double (&r)[NF][K]) {
    const double* pbco = pb;
    const double* pbci = pb + 16;
    double s0[NF], s1[NF], o0[NF], o1[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) { s0[f] = 0.0; s1[f] = 0.0; o0[f] = 0.0; o1[f] = 0.0; }
#pragma unroll 1
    for (int i = 0; i < kLmd; i++) {
        double v[NF];
        row(end, i, v);
#pragma unroll
        for (int f = 0; f < NF; f++) { s0[f] += pbci[i] * v[f]; s1[f] += pbci[kLmd + i] * v[f]; }
        row(1 - end, i, v);
#pragma unroll
        for (int f = 0; f < NF; f++) { o0[f] += pbco[i] * v[f]; o1[f] += pbco[kLmd + i] * v[f]; }
    }
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const double a = s0[f] + o0[f], b = s1[f] + o1[f];
        if (end == 0) {
            r[f][0] = a;
            r[f][1] = b;
        } else {
#pragma unroll
            for (int t = 0; t < K; t++) {
                if (t == L - 1) r[f][t] = -a;
                if (t == L - 2) r[f][t] = -b;
            }
        }
    }
}

// characteristic correction of a face (first or last chunk of a line, never
// both: lines have at least two chunks), weighted by sbcc on the kMbci rows
// next to the face; the face derivative is the uncorrected solve result.  L =
// rows of the chunk.
template <int K, int NF, class SW, class FACE>
__device__ __forceinline__ void face_correction(const SW& sw, const FACE& fc, int face, int L, double (&r)[NF][K]) {
    static_assert(kMbci == 1, "the face row only");
    double drv[NF], corr[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        drv[f] = r[f][0];
#pragma unroll
        for (int t = 1; t < K; t++)
            if (face && t == L - 1) drv[f] = r[f][t];
    }
    sw.gcbc(fc, face, drv, corr);
#pragma unroll
    for (int t = 0; t < K; t++)
        if (face ? t == L - 1 : t == 0) {
#pragma unroll
            for (int f = 0; f < NF; f++) r[f][t] += fc.w * corr[f];
        }
}

// functors that reduce the time step's maxima: value = in the point
// evaluation of a y/z sweep (constant metrics), close = in the closing x
// sweep's stores (per-point metrics)
template <class SW, class = void>
struct DtFold {
    static constexpr bool value = false;
    static constexpr bool close = false;
};
template <class SW>
struct DtFold<SW, std::void_t<decltype(SW::kDt)>> {
    static constexpr bool value = SW::kDt && !SW::kCurv;
    static constexpr bool close = SW::kDt && SW::kCurv;
};

// Many operators in one launch (batched subdomains): a direct or x kernel
// launched with a BatchItems argument takes its descriptor from operator
// items[i].x and runs that operator's workgroup items[i].y, items round-robin
// over the grid.  Without one these are no-ops.
template <class SW>
struct BatchOp {
    AxisDesc ax;
    SweepCommon cm;
    SW sw;
};
template <class SW>
struct BatchItems {
    const BatchOp<SW>* ops;
    const int2* items;
    int n;
    __device__ __forceinline__ bool more(int& it) const { return (it += gridDim.x) < n; }
    // the operator is the same for the whole workgroup: into scalar registers
    // word by word, as a by-value kernel argument is
    __device__ __forceinline__ void take(int it, AxisDesc& ax, SweepCommon& cm, SW& sw, long& group) const {
        static_assert(sizeof(BatchOp<SW>) % 4 == 0, "moves as 32-bit words");
        constexpr int kWords = sizeof(BatchOp<SW>) / 4;
        const unsigned* src =
            reinterpret_cast<const unsigned*>(ops + __builtin_amdgcn_readfirstlane(items[it].x));
        group = __builtin_amdgcn_readfirstlane(items[it].y);
        unsigned words[kWords];
#pragma unroll
        for (int i = 0; i < kWords; i++) words[i] = __builtin_amdgcn_readfirstlane(src[i]);
        BatchOp<SW> o;
        __builtin_memcpy(&o, words, sizeof o);
        ax = o.ax;
        cm = o.cm;
        sw = o.sw;
    }
};
struct NoBatch {
    __device__ __forceinline__ bool more(int&) const { return false; }
    template <class SW>
    __device__ __forceinline__ void take(int, AxisDesc& ax, SweepCommon&, SW&, long& group) const {
        group = group_of(ax.xcd);
    }
};

// ---------------------------------------------------------------------------
// variant "direct", y/z lines: TL consecutive lines x P chunks per workgroup;
// each thread evaluates the pointwise inputs of its own K rows once, the halo
// rows on each side and the 8 + 8 rows of a periodic seam come from the other
// chunks through LDS.
//
// Bound by memory latency at the occupancy its registers allow (K = 16: 256
// VGPRs, 8 waves a CU): the K x NF values stay in registers from the loads to
// the stores.  So nothing but them is live: the loads run kRowsAhead rows ahead
// of the evaluation (all rows at once spill 500-700 B a lane), a field's window
// exists only while its right-hand side is formed, and the epilogue's loads run
// kRowsOut rows ahead of the additions.  Measured at 256^3 (us, before -> now;
// a copy of 2.1 GB runs at 4.8 TB/s, the same row pattern without arithmetic
// at 5.3 along y and 4.7 along z): S1y 284 -> 220 (5.5 TB/s), S2y 550 -> 482
// (5.3), S1z 309 -> 259 (4.7), S2z 514 -> 400 (4.7).
// ---------------------------------------------------------------------------
constexpr int kRowsAhead = 2;   // rows whose loads are in flight while a row is evaluated
constexpr int kRowsOut = 4;     // rows whose epilogue loads are in flight

template <int K, int AX, int TL, class SW, bool GCBC, bool EX, bool NT, class BATCH = NoBatch>
__global__ void __launch_bounds__(TL == 32 ? 512 : TL * kMaxP < 1024 ? TL * kMaxP : 1024)
__attribute__((amdgpu_waves_per_eu(K == 16 ? SW::kWpe16 : SW::kWpe)))
direct_kernel(AxisDesc ax, SweepCommon cm, SW sw, BATCH batch) {
    extern __shared__ double lds[];       // direct_lds
    constexpr int NF = SW::NF;
    constexpr int H = SW::kH;
    constexpr int W = K + 2 * H;
    static_assert(AX != 0, "x lines run xt_kernel");
    static_assert(H <= K, "halo rows come from the neighbouring chunks only");
    int it = blockIdx.x;
    do {
    long group;
    batch.take(it, ax, cm, sw, group);

    const int N = ax.N, P = ax.P, NP = P * K;
    const Chunks<K, EX> ch(N, P);
    const int lloc = threadIdx.x % TL;
    // 64 lines: one chunk a wave, its table entries come by scalar loads
    const int c = TL == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / TL) : threadIdx.x / TL;
    const long line = group * TL + lloc;
    const bool act = line < ax.nlines;
    const int s = c * K, row0 = ch.start(c);      // table and line position of the chunk
    const bool whole = ch.whole(c);
    const uoff st = (uoff)ax.st * 8u;
    // threads past the last line repeat it, padding rows repeat the chunk's last
    // row: no branches around the loads, and nothing of theirs is stored
    const uoff base = line_off(AX, (uoff)(act ? line : ax.nlines - 1), (uoff)cm.lxi, (uoff)cm.plane);
    const uoff cbase = base + (uoff)row0 * st;
    auto off = [&](int t) { return cbase + (uoff)(EX || t < K - 1 || whole ? t : K - 2) * st; };
    const double* tab = SW::kFilter ? ax.ftab : ax.tab;
    const bool cyc = SW::kFilter && ax.seam;
    const bool first = c == 0, last = c == P - 1;

    // time-step maxima (DtFold functors; every lane of the workgroup's waves
    // is a thread, the launcher checks)
    constexpr bool kDt = DtFold<SW>::value;
    double dm0 = 0.0, dm1 = 0.0;
    double x[NF][K];
    // the loads of kRowsAhead rows are in flight while a row is evaluated
    constexpr int RA = NF > 1 && kRowsAhead < K ? kRowsAhead : K;
    typename SW::Raw raw[RA];
#pragma unroll
    for (int t = 0; t < RA; t++) sw.template load<NT>(off(t), raw[t]);
    if (RA < K) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < K; t++) {
        double v[NF];
        if constexpr (kDt) sw.eval_dt(raw[t % RA], v, dm1);
        else sw.eval(raw[t % RA], v);
#pragma unroll
        for (int f = 0; f < NF; f++) x[f][t] = v[f];
        if (t + RA < K) {
            sw.template load<NT>(off(t + RA), raw[t % RA]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if constexpr (kDt) {
        // the convective maximum from u, v, w, c^2 of the rows; the viscous one
        // at the largest 1/rho
#pragma unroll
        for (int t = 0; t < K; t++) dm0 = fmax(dm0, dt_conv(sw.ph, x[0][t], x[1][t], x[2][t], x[3][t]));
        dm1 = dt_visc(sw.ph, dm1);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            dm0 = fmax(dm0, __shfl_xor(dm0, o));
            dm1 = fmax(dm1, __shfl_xor(dm1, o));
        }
    }
    // halo rows through LDS, hb[(f*2H + k)*P + c][TL], k = the first H then the
    // last H rows of chunk c, FX fields at a time (neighbours wrap on cyclic
    // lines); on a seam axis also the 8 rows next to each end, [2 end][8][NF][TL]
    constexpr int FX = SW::kFilter ? 1 : NF;
    const int cl = c > 0 ? c - 1 : (cyc ? P - 1 : 0), cr = c + 1 < P ? c + 1 : (cyc ? 0 : P - 1);
    double* ends = lds + 2 * H * NF * P * TL;
    double r[NF][K];
#pragma unroll
    for (int f0 = 0; f0 < NF; f0 += FX) {
        if (f0 > 0) __syncthreads();
#pragma unroll
        for (int e = 0; e < FX; e++) {
            const int f = f0 + e;
#pragma unroll
            for (int k = 0; k < H; k++) {
                lds[((e * 2 * H + k) * P + c) * TL + lloc] = x[f][k];
                lds[((e * 2 * H + H + k) * P + c) * TL + lloc] =
                    whole ? x[f][K - H + k] : x[f][K - H + k > 0 ? K - H + k - 1 : 0];
            }
        }
        if (!SW::kFilter && ax.seam && (first || last)) {
#pragma unroll
            for (int i = 0; i < kLmd; i++)
#pragma unroll
                for (int f = 0; f < NF; f++)
                    ends[(((first ? 0 : kLmd) + i) * NF + f) * TL + lloc] = first ? x[f][i] : x[f][K - 1 - i];
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < FX; e++) {
            const int f = f0 + e;
            double w[W], right[H];
#pragma unroll
            for (int k = 0; k < H; k++) {
                w[k] = lds[((e * 2 * H + H + k) * P + cl) * TL + lloc];
                right[k] = lds[((e * 2 * H + k) * P + cr) * TL + lloc];
            }
#pragma unroll
            for (int t = 0; t < K; t++) w[t + H] = x[f][t];
            close_window<K, H, W>(w, right, whole);
            if constexpr (SW::kFilter) filter_rhs<K, W>(w, r[f], first && !cyc, last && !cyc, ax.ftab + 6 * NP + 8);
            else window_rhs<K, W>(w, r[f], first && !ax.seam, last && !ax.seam);
        }
    }
    if (!SW::kFilter && ax.seam && (first || last))
        seam_rows<K, NF>([&](int end, int i, double* v) {
#pragma unroll
            for (int f = 0; f < NF; f++) v[f] = ends[((end * kLmd + i) * NF + f) * TL + lloc];
        }, first ? 0 : 1, K, cm.pb, r);

    double carry[NF], G[NF], X[NF];
    forward_local<K, NF>(tab, NP, s, r, carry);
    __syncthreads();                                // halo reads done: reuse LDS
#pragma unroll
    for (int f = 0; f < NF; f++) lds[(f * P + c) * TL + lloc] = carry[f];
    // the waves' time-step maxima go past the carries of both folds
    double* dl = lds + 3 * NF * P * TL;
    if constexpr (kDt) {
        if ((threadIdx.x & 63) == 0) {
            dl[2 * (threadIdx.x >> 6)] = dm0;
            dl[2 * (threadIdx.x >> 6) + 1] = dm1;
        }
    }
    __syncthreads();
    if constexpr (kDt) {
        if (threadIdx.x == 0) {
            double a0 = 0.0, a1 = 0.0;
            for (int v = 0; v < (int)(blockDim.x >> 6); v++) {
                a0 = fmax(a0, dl[2 * v]);
                a1 = fmax(a1, dl[2 * v + 1]);
            }
            sw.dtpart[2 * blockIdx.x] = a0;
            sw.dtpart[2 * blockIdx.x + 1] = a1;
        }
    }
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
    if (cyc) {
        // rows 0 and N-1 of the modified system through LDS (after the folds' reads)
        double* ends = lds + 2 * NF * P * TL;
        if (first) {
#pragma unroll
            for (int f = 0; f < NF; f++) ends[f * TL + lloc] = r[f][0];
        }
        if (last) {
#pragma unroll
            for (int f = 0; f < NF; f++) ends[(NF + f) * TL + lloc] = r[f][K - 1];
        }
        __syncthreads();
        double y0[NF], yN1[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) {
            y0[f] = ends[f * TL + lloc];
            yN1[f] = ends[(NF + f) * TL + lloc];
        }
        cyclic_correction<K, NF>(tab, NP, s, y0, yN1, r);
    }

    if (act) {
    if constexpr (SW::kEnds) {
        if (first) sw.end_value(0, line, r[0][0]);
        if (last) sw.end_value(1, line, r[0][K - 1]);
    }
    if constexpr (GCBC) {
        if (first || last) {
            const auto fc = sw.face_in(base + (uoff)(first ? 0 : N - 1) * st, first ? 0 : 1, cm.sbcc);
            face_correction<K, NF, SW>(sw, fc, first ? 0 : 1, K, r);
        }
    }
    // every row's epilogue loads before the first store, kRowsOut rows in flight
    if constexpr (SW::kAdds) {
        typename SW::Out out[kRowsOut];
#pragma unroll
        for (int t = 0; t < kRowsOut; t++) sw.template load_out<NT>(off(t), out[t]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < K; t++) {
            double d[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) d[f] = r[f][t];
            sw.add_out(out[t % kRowsOut], d);
#pragma unroll
            for (int f = 0; f < NF; f++) r[f][t] = d[f];
            if (t + kRowsOut < K) {
                sw.template load_out<NT>(off(t + kRowsOut), out[t % kRowsOut]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < K; t++) {
        if (EX || t < K - 1 || whole) {
            double d[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) d[f] = r[f][t];
            sw.template store<NT>(off(t), d);
        }
    }
    }
    if constexpr (!std::is_same_v<BATCH, NoBatch>) __syncthreads();      // the LDS is free for the next item
    } while (batch.more(it));
}

// ---------------------------------------------------------------------------
// variant "direct" for x lines: one wave holds the P chunks of 64/P
// consecutive lines (lane = line * P + chunk), one contiguous run of memory.
// Lanes load and evaluate that run with fully coalesced accesses (K points
// per lane), the values are transposed field by field through a wave-private
// LDS buffer into the chunk layout (halo and seam rows included), the line is
// solved with wave scans, and the results go back through the buffer for
// coalesced stores.  No workgroup barrier: a workgroup is one wave.
//
// Two waves a SIMD, each with its 8 points' loads in flight; at 256^3 the
// sweeps run at the rate of a plain stream of the same fields (5.6 TB/s): S1x
// 556 -> 418 us (144 bytes a point instead of 176), filter 392 -> 237, S2x 606
// -> 528 in a step.  What held them back were instructions, not bytes (the
// filter: 4150 a wave, 2000 now): branches around every point, closure rows
// tested row by row, seam rows read again from memory.
// ---------------------------------------------------------------------------
template <int K, class SW, bool GCBC, bool EX, bool NT, class BATCH = NoBatch>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
xt_kernel(AxisDesc ax, SweepCommon cm, SW sw, BATCH batch) {
    extern __shared__ double lds[];       // xt_lds
    constexpr int NF = SW::NF;
    constexpr int J = K;                  // points per lane: (64/P)*N <= 64*K
    constexpr int H = SW::kH;
    constexpr int W = K + 2 * H;
    constexpr int LK = K == 8 ? 3 : 4;
    static_assert(K == 8 || K == 16, "chunks of 8 or 16 points");
    int it = blockIdx.x;
    do {
    long group;
    batch.take(it, ax, cm, sw, group);
    // lds: [64/P lines][P chunks][K+1], 64 slots for lanes past the run, then
    // (kStash > 0) the stashed point values [kStash][J][64]

    const int N = ax.N, P = ax.P, NP = P * K;
    const Chunks<K, EX> ch(N, P);
    const int lane = threadIdx.x;
    const int lpw = 64 / P;
    double* stash = lds + lpw * P * (K + 1) + 64;
    const long line0 = group * lpw;
    const int nl = (int)min((long)lpw, ax.nlines - line0);   // lines of this wave
    const int npts = nl * N;
    const uoff run = line_off(0, (uoff)line0, (uoff)cm.lxi, (uoff)cm.plane);
    // lanes past the run repeat its last point: no branches around the loads
    auto off = [&](int j) { return run + (uoff)min(lane + 64 * j, npts - 1) * 8u; };

    // coalesced evaluation: lane handles points lane + 64*j of the run.  A
    // functor with too many values a point for all 8 in flight (kBlocks) takes
    // one after the other: a branch a point keeps the compiler from hoisting
    // the next ones' loads (S2C: 8 points at once spill 580 B a lane, 233 -> 541 us)
    double xq[NF][J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        double x[NF];
        if (!SW::kBlocks || lane + 64 * j < npts) {
            point<NT>(sw, off(j), x);
        } else {
#pragma unroll
            for (int f = 0; f < NF; f++) x[f] = 0.0;
        }
#pragma unroll
        for (int f = 0; f < NF; f++) xq[f][j] = x[f];
    }
    const int li = lane / P, c = lane % P;
    const bool work = li < nl;
    const int lr = work ? li : 0;
    const int s = c * K;
    const bool first = c == 0, last = c == P - 1, whole = ch.whole(c);
    const double* tab = SW::kFilter ? ax.ftab : ax.tab;
    const bool cyc = SW::kFilter && ax.seam;
    if constexpr (SW::kStash > 0) {
        // lane-contiguous: no bank conflicts; each lane reads back only its own slots
#pragma unroll
        for (int f = 0; f < SW::kStash; f++)
#pragma unroll
            for (int j = 0; j < J; j++) stash[(f * J + j) * 64 + lane] = xq[f][j];
    }

    // LDS slot of each of the lane's points: chunk * (K+1) + row of the chunk
    auto whole_slot = [](int row) { return (row >> LK) * (K + 1) + (row & (K - 1)); };
    auto row_slot = [&](int row) {
        const int q = row - K;                                   // rows after the first chunk
        const int cs = (q * (65536 / (K - 1) + 1)) >> 16;        // q / (K-1), exact for q < 1024
        if (row < K) return row;
        return q < (K - 1) * ch.D ? (cs + 1) * (K + 1) + (q - cs * (K - 1)) : whole_slot(row + ch.D);
    };
    int slot[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int p = lane + 64 * j;
        if (EX) {
            slot[j] = whole_slot(p);
        } else {
            // p / N by the reciprocal rounded up: exact for p < 1024, N <= 1024
            const int l = (int)(((unsigned)p * ((0x1000000u + N - 1) / (unsigned)N)) >> 24);
            slot[j] = xt_slot<K>(l, P, 0, 0) + row_slot(p - l * N);
        }
        if (p >= npts) slot[j] = lpw * P * (K + 1) + lane;
    }

    // halo chunks: the neighbours, wrapped on a cyclic line (other lines clamp;
    // their values there are not used)
    const int hl = c > 0 ? c - 1 : (cyc ? P - 1 : 0);
    const int hr = c + 1 < P ? c + 1 : (cyc ? 0 : P - 1);
    const int left = xt_slot<K>(lr, P, hl, K - H) - (ch.whole(hl) ? 0 : 1);

    double r[NF][K];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; j++) lds[slot[j]] = xq[f][j];
        __syncthreads();
        double w[W], right[H];
#pragma unroll
        for (int u = 0; u < H; u++) {
            w[u] = lds[left + u];
            right[u] = lds[xt_slot<K>(lr, P, hr, u)];
        }
#pragma unroll
        for (int t = 0; t < K; t++) w[t + H] = lds[xt_slot<K>(lr, P, c, t)];
        close_window<K, H, W>(w, right, whole);
        if constexpr (SW::kFilter) {
            filter_rhs<K, W>(w, r[f], first && !cyc, last && !cyc, ax.ftab + 6 * NP + 8);
        } else {
            window_rhs<K, W>(w, r[f], first && !ax.seam, last && !ax.seam);
            // both ends of the line are in the buffer; one pass serves the lanes of both
            if (ax.seam && (first || last)) {
                double rf[1][K];
#pragma unroll
                for (int t = 0; t < K; t++) rf[0][t] = r[f][t];
                seam_rows<K, 1>([&](int end, int i, double* v) {
                    v[0] = lds[end ? xt_slot<K>(lr, P, P - 1, K - 1 - i) : xt_slot<K>(lr, P, 0, i)];
                }, first ? 0 : 1, K, cm.pb, rf);
#pragma unroll
                for (int t = 0; t < K; t++) r[f][t] = rf[0][t];
            }
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
    if (cyc) {
        double y0[NF], yN1[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) {
            y0[f] = __shfl(r[f][0], lr * P);
            yN1[f] = __shfl(r[f][K - 1], lr * P + P - 1);
        }
        cyclic_correction<K, NF>(tab, NP, s, y0, yN1, r);
    }
    if constexpr (SW::kEnds) {
        if (work && first) sw.end_value(0, line0 + li, r[0][0]);
        if (work && last) sw.end_value(1, line0 + li, r[0][K - 1]);
    }
    if constexpr (GCBC) {
        if (work && (first || last)) {
            const auto fc = sw.face_in(run + (uoff)(lr * N + (first ? 0 : N - 1)) * 8u, first ? 0 : 1, cm.sbcc);
            face_correction<K, NF, SW>(sw, fc, first ? 0 : 1, K, r);
        }
    }

    // back to the coalesced layout, one field at a time
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
    double mm[2] = {0.0, 0.0};           // DtFold<SW>::close: the time step's maxima
    // every point's epilogue loads before the first store
    if constexpr (SW::kAdds) {
#pragma unroll
        for (int j = 0; j < J; j++) {
            if (!SW::kBlocks || lane + 64 * j < npts) {
                double d[NF];
#pragma unroll
                for (int f = 0; f < NF; f++) d[f] = xo[f][j];
                add_out<NT>(sw, off(j), d);
#pragma unroll
                for (int f = 0; f < NF; f++) xo[f][j] = d[f];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; j++) {
        if (lane + 64 * j < npts) {
            double d[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) d[f] = xo[f][j];
            if constexpr (SW::kStash > 0) {
                double sv[SW::kStash > 0 ? SW::kStash : 1];
#pragma unroll
                for (int f = 0; f < SW::kStash; f++) sv[f] = stash[(f * J + j) * 64 + lane];
                if constexpr (DtFold<SW>::close) sw.template store_pv_dt<NT>(off(j), d, sv, mm);
                else sw.template store_pv<NT>(off(j), d, sv);
            } else {
                sw.template store<NT>(off(j), d);
            }
        }
    }
    if constexpr (DtFold<SW>::close) {
        // the workgroup is one wave: reduce across it, one pair per workgroup
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            mm[0] = fmax(mm[0], __shfl_xor(mm[0], o));
            mm[1] = fmax(mm[1], __shfl_xor(mm[1], o));
        }
        if (lane == 0) {
            sw.dtpart[2 * blockIdx.x] = mm[0];
            sw.dtpart[2 * blockIdx.x + 1] = mm[1];
        }
    }
    if constexpr (!std::is_same_v<BATCH, NoBatch>) __syncthreads();
    } while (batch.more(it));
}

// ---------------------------------------------------------------------------
// variant "tile": the pointwise inputs of TL lines pass through an LDS tile
// one row block (kCB chunks + halo) at a time with coalesced loads -- every
// point is evaluated once -- and chunk threads stream their windows from the
// tile.  The tile memory is then reused for the carries and, for x lines, for
// a transposed coalesced store.
// ---------------------------------------------------------------------------
constexpr int kCB = 8;   // chunks per row block

template <int K>
__host__ __device__ constexpr int tile_rows() { return kCB * K + 4; }

template <int K, int AX, int TL, class SW, bool GCBC>
__global__ void __launch_bounds__(TL * kMaxP) tile_kernel(AxisDesc ax, SweepCommon cm, SW sw) {
    constexpr int NF = SW::NF;
    constexpr int TLP = TL + 1;
    constexpr int RB = tile_rows<K>();
    extern __shared__ double lds[];    // tile [NF][RB][TLP]

    const int N = ax.N, P = ax.P, NP = P * K;
    const int nthr = TL * P;
    const int tid = threadIdx.x;
    const int lloc = tid % TL, c = tid / TL;
    const long line0 = group_of(ax.xcd) * TL;
    const long line = line0 + lloc;
    const bool act = line < ax.nlines;
    const int s = chunk_start(N, P, K, c), L = chunk_start(N, P, K, c + 1) - s;
    const uoff st = (uoff)ax.st * 8u;
    const uoff lxi = (uoff)cm.lxi, plane = (uoff)cm.plane;
    const uoff base = line_off(AX, act ? (uoff)line : 0u, lxi, plane);
    const double* tab = ax.tab;
    const int nb = (P + kCB - 1) / kCB;

    double r[NF][K];
    for (int b = 0; b < nb; b++) {
        const int c0 = b * kCB, c1 = min(P, c0 + kCB);
        const int rs = max(0, chunk_start(N, P, K, c0) - 2);
        const int re = min(N, chunk_start(N, P, K, c1) + 2);
        const int nrows = re - rs;
        if (b > 0) __syncthreads();
        for (int p = tid; p < TL * nrows; p += nthr) {
            int l, row;
            if (AX == 0) { l = p / nrows; row = rs + p % nrows; }
            else         { l = p % TL;    row = rs + p / TL; }
            const long ln = line0 + l;
            double x[NF];
            if (ln < ax.nlines) {
                point<false>(sw, line_off(AX, (uoff)ln, lxi, plane) + (uoff)row * st, x);
            } else {
#pragma unroll
                for (int f = 0; f < NF; f++) x[f] = 0.0;
            }
#pragma unroll
            for (int f = 0; f < NF; f++) lds[(f * RB + row - rs) * TLP + l] = x[f];
        }
        __syncthreads();
        if (c >= c0 && c < c1) {
            auto row_of = [&](int u, double* x) {
                const int row = s - 2 + u;
                const bool in = row >= 0 && row < N;
#pragma unroll
                for (int f = 0; f < NF; f++) x[f] = in ? lds[(f * RB + row - rs) * TLP + lloc] : 0.0;
            };
            stream_rhs<K, NF>(row_of, r, s, L, N, ax.seam);
        }
    }
    if (act && ax.seam && (c == 0 || c == P - 1))
        seam_rows<K, NF>([&](int end, int i, double* v) { point<false>(sw, base + (uoff)(end ? N - 1 - i : i) * st, v); },
                         c == 0 ? 0 : 1, L, cm.pb, r);

    double carry[NF], G[NF], X[NF];
    forward_local<K, NF>(tab, NP, c * K, r, carry);
    __syncthreads();                                   // tile reads done: reuse for carries
#pragma unroll
    for (int f = 0; f < NF; f++) lds[(f * P + c) * TL + lloc] = carry[f];
    __syncthreads();
    fold_forward<NF, K>(lds, tab, NP, P, TL, c, lloc, G);
    apply_carry<K, NF>(tab, 3 * NP, c * K, r, G);
#pragma unroll
    for (int t = 1; t < K; t++)
#pragma unroll
        for (int f = 0; f < NF; f++) r[f][t] = t < L ? r[f][t] : 0.0;
    backward_local<K, NF>(tab, NP, c * K, r, carry);
    double* xb = lds + NF * P * TL;
#pragma unroll
    for (int f = 0; f < NF; f++) xb[(f * P + c) * TL + lloc] = carry[f];
    __syncthreads();
    fold_backward<NF, K>(xb, tab, NP, P, TL, c, lloc, X);
    apply_carry<K, NF>(tab, 4 * NP, c * K, r, X);

    if constexpr (GCBC) {
        if (act && (c == 0 || c == P - 1)) {
            const auto fc = sw.face_in(base + (uoff)(c == 0 ? 0 : N - 1) * st, c == 0 ? 0 : 1, cm.sbcc);
            face_correction<K, NF, SW>(sw, fc, c == 0 ? 0 : 1, L, r);
        }
    }

    if (AX != 0) {
        if (!act) return;
#pragma unroll
        for (int t = 0; t < K; t++) {
            if (t < L) {
                double d[NF];
#pragma unroll
                for (int f = 0; f < NF; f++) d[f] = r[f][t];
                add_out<false>(sw, base + (uoff)(s + t) * st, d);
#pragma unroll
                for (int f = 0; f < NF; f++) r[f][t] = d[f];
            }
        }
#pragma unroll
        for (int t = 0; t < K; t++) {
            if (t < L) {
                double d[NF];
#pragma unroll
                for (int f = 0; f < NF; f++) d[f] = r[f][t];
                sw.template store<false>(base + (uoff)(s + t) * st, d);
            }
        }
        return;
    }
    // x lines: results back through the tile, one row block at a time, stored along the line
    for (int b = 0; b < nb; b++) {
        const int c0 = b * kCB, c1 = min(P, c0 + kCB);
        const int rs = chunk_start(N, P, K, c0);
        const int re = chunk_start(N, P, K, c1);
        const int nrows = re - rs;
        __syncthreads();
        if (c >= c0 && c < c1) {
#pragma unroll
            for (int t = 0; t < K; t++)
                if (t < L)
#pragma unroll
                    for (int f = 0; f < NF; f++) lds[(f * RB + s + t - rs) * TLP + lloc] = r[f][t];
        }
        __syncthreads();
        for (int p = tid; p < TL * nrows; p += nthr) {
            const int l = p / nrows, row = rs + p % nrows;
            const long ln = line0 + l;
            if (ln >= ax.nlines) continue;
            double d[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) d[f] = lds[(f * RB + row - rs) * TLP + l];
            const uoff bo = line_off(AX, (uoff)ln, lxi, plane) + (uoff)row * st;
            add_out<false>(sw, bo, d);
            sw.template store<false>(bo, d);
        }
    }
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------
// the descriptor a launch of `groups` workgroups runs with: its xcd field
// becomes the run length code of group_of, runs of at most `most` groups
inline AxisDesc with_runs(const AxisDesc& ax, long groups, bool on, int most) {
    AxisDesc a = ax;
    a.xcd = 0;
    if (on) {
        a.xcd = 1;
        while ((2L << (a.xcd - 1)) <= most && (16L << (a.xcd - 1)) <= groups) a.xcd++;
    }
    return a;
}

// Streaming hints pay once a sweep passes over more than the 256 MB of the
// last-level cache (below, the next sweep finds there what this one wrote:
// 128^3 S2y 60 us without them against 71 with; above, 256^3 S2z 455 against
// 526), and only where a row access covers whole cache lines: with rows off
// the 128-byte grid a line is shared by two workgroups (201x160x176: S2y 323
// against 366 us, S1x 214 against 243).  x lines are one run of memory, of
// which only the ends are shared; rows of 16 bytes already pay there.
// kBytes is the memory a point of the sweep takes, a field read and written
// once, times the fields over grid.y (five-field derivatives of the
// per-operator right-hand side at 192^3: 1932 -> 1897 us a right-hand side
// against counting one of them; counting the transposed filter's fields
// twice: 160^3 adjoint 2393 -> 2414).
template <class SW>
static bool streams(const AxisDesc& ax, const SweepCommon& cm, unsigned gy) {
    const int align = ax.st == 1 ? 2 : 16;
    return cm.lxi % align == 0 && (double)SW::kBytes * gy * (double)ax.N * (double)ax.nlines > 256.0 * (1 << 20);
}

template <int K, class SW, bool GCBC>
static const void* xt_symbol(bool exact, bool nt) {
    if (exact) return nt ? (const void*)xt_kernel<K, SW, GCBC, true, true> : (const void*)xt_kernel<K, SW, GCBC, true, false>;
    return nt ? (const void*)xt_kernel<K, SW, GCBC, false, true> : (const void*)xt_kernel<K, SW, GCBC, false, false>;
}

// Lines a workgroup of a y/z sweep takes where tl (8 or 16) asks for 16.
// One field on lines of up to 16 chunks: 64, so that a wave is one chunk, its
// table entries come by scalar loads and rows are 512 bytes (256^3 filter y 309 ->
// 283, z 316 -> 292 us; 128^3 40 -> 34, 40 -> 36).  The five- and four-field
// sweeps along z on up to 16 chunks of 16 points: 32, 256-byte rows of a plane
// that is otherwise passed over in 128-byte pieces (256^3 S2z 442 -> 415, S1z
// 271 -> 269 us, with FP32 storage 412 -> 351, 299 -> 208; 128^3 S2z 47 -> 43,
// S1z 28 -> 25; over lengths of 48 to 256 a right-hand side gains 1 % on
// average, 8 % at most, and loses 1 to 3 % at 9, 10, 13 and 15 chunks, which
// leave waves of a CU empty).  Along y, where 16 lines' rows lie next to the
// following workgroup's, 32 lose (S2y 484 -> 546, S1y 218 -> 247 us).
template <int K, int AX, class SW>
static int block_lines(int P, int tl) {
    if (tl == 8) return 8;
    if (SW::NF == 1 && P <= 16) return 64;
    return AX == 2 && K == 16 && SW::NF > 1 && !SW::kFilter && P <= 16 ? 32 : 16;
}

template <int K, int AX, int TL, class SW, bool GCBC>
static const void* direct_at(bool exact, bool nt) {
    if (exact) return nt ? (const void*)direct_kernel<K, AX, TL, SW, GCBC, true, true>
                         : (const void*)direct_kernel<K, AX, TL, SW, GCBC, true, false>;
    return nt ? (const void*)direct_kernel<K, AX, TL, SW, GCBC, false, true>
              : (const void*)direct_kernel<K, AX, TL, SW, GCBC, false, false>;
}

// 8 lines a workgroup are 64-byte rows: never streamed
template <int K, int AX, class SW, bool GCBC>
static const void* direct_symbol(int TL, bool exact, bool nt) {
    if (TL == 8) return exact ? (const void*)direct_kernel<K, AX, 8, SW, GCBC, true, false>
                              : (const void*)direct_kernel<K, AX, 8, SW, GCBC, false, false>;
    if constexpr (SW::NF == 1)
        if (TL == 64) return direct_at<K, AX, 64, SW, GCBC>(exact, nt);
    if constexpr (AX == 2 && K == 16 && SW::NF > 1 && !SW::kFilter)
        if (TL == 32) return direct_at<K, AX, 32, SW, GCBC>(exact, nt);
    return direct_at<K, AX, 16, SW, GCBC>(exact, nt);
}

template <class SW, class BATCH = NoBatch>
static int launch(const void* k, dim3 grid, dim3 block, size_t lds, AxisDesc a, SweepCommon cm, SW sw, hipStream_t s,
                  BATCH batch = BATCH()) {
    if (lds > 65536) CS_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    void* args[] = {&a, &cm, &sw, &batch};
    CS_HIP(hipLaunchKernel(k, grid, block, args, lds, s));
    return CS_OK;
}

// LDS of a workgroup
template <int K, class SW>
static size_t xt_lds(int P) { return sizeof(double) * ((64 / P) * P * (K + 1) + 64 + SW::kStash * K * 64); }
template <class SW>
static size_t direct_lds(int P, int TL, bool seam) {
    const size_t halo = (size_t)(SW::kFilter ? 1 : SW::NF) * 2 * SW::kH * P + (!SW::kFilter && seam ? SW::NF * 2 * kLmd : 0);
    const size_t carries = (size_t)2 * SW::NF * P + (SW::kFilter ? 2 * SW::NF : 0);
    return sizeof(double) * TL * (halo > carries ? halo : carries);
}

// x sweeps: a workgroup is the 64/P lines of one wave, runs of 64 an XCD
// (measured 4.8 -> 5.3 TB/s for a copy of that shape)
template <int K, class SW, bool GCBC>
static int launch_x(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, unsigned gy, hipStream_t s) {
    const int lpw = 64 / ax.P;
    const size_t lds = xt_lds<K, SW>(ax.P);
    const dim3 grid((unsigned)((ax.nlines + lpw - 1) / lpw), gy);
    return launch(xt_symbol<K, SW, GCBC>(ax.N == ax.P * K, streams<SW>(ax, cm, gy)), grid, dim3(64), lds,
                  with_runs(ax, grid.x, true, 64), cm, sw, s);
}

// y/z sweeps: TL lines a workgroup; along y runs of 128 neighbouring lines an
// XCD, along z of 1024 (256^3: S1y 240 -> 216, S2y 529 -> 485, S2z 488 -> 440,
// S1z 318 -> 279 us against plain order)
template <int K, int AX, class SW, bool GCBC>
static int launch_yz(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, int TL, bool runs, size_t lds,
                     unsigned gy, hipStream_t s) {
    const dim3 grid((unsigned)((ax.nlines + TL - 1) / TL), gy);
    return launch(direct_symbol<K, AX, SW, GCBC>(TL, ax.N == ax.P * K, streams<SW>(ax, cm, gy)), grid, dim3(TL * ax.P),
                  lds, with_runs(ax, grid.x, runs, (AX == 1 ? 128 : 1024) / TL), cm, sw, s);
}

template <int K, int AX, class SW, bool GCBC>
static int launch_sweep(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, hipStream_t s) {
    constexpr int NF = SW::NF;
    if constexpr (K == 8) {
        // the tiles take any chunk lengths
        if (ax.variant == 1 || !chunks_fit(ax.N, ax.P, K)) {
            const size_t tile = (size_t)NF * tile_rows<K>() * (ax.tl + 1);
            const size_t carries = (size_t)2 * NF * ax.P * ax.tl;
            const size_t lds = sizeof(double) * (tile > carries ? tile : carries);
            const dim3 grid((unsigned)((ax.nlines + ax.tl - 1) / ax.tl));
            return launch(ax.tl == 8 ? (const void*)tile_kernel<K, AX, 8, SW, GCBC>
                                     : (const void*)tile_kernel<K, AX, 16, SW, GCBC>,
                          grid, dim3(ax.tl * ax.P), lds, with_runs(ax, grid.x, ax.xcd, 64), cm, sw, s);
        }
    }
    if constexpr (AX == 0) {
        static_assert(K == 8, "x lines run 8-point chunks");
        return launch_x<K, SW, GCBC>(ax, cm, sw, 1u, s);
    } else {
        const int TL = block_lines<K, AX, SW>(ax.P, ax.tl);
        return launch_yz<K, AX, SW, GCBC>(ax, cm, sw, TL, ax.xcd != 0, direct_lds<SW>(ax.P, TL, ax.seam), 1u, s);
    }
}

// the filter sweep on chunks of K points (8 along x; 8 or 16 along y/z, the
// axis's filter descriptor); SW = SF<AX> (five variables per workgroup)
// or SF1<AX> (one variable per workgroup, grid.y = 5)
template <int K, int AX, class SW>
static int launch_filter(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, hipStream_t s) {
    constexpr int NF = SW::NF;
    static_assert(AX != 0 || K == 8, "x filter sweeps run 8-point chunks");
    const unsigned gy = NF == 1 ? 5u : 1u;
    if (ax.K != K || !ax.ftab) return fail(CS_ERR_STATE, "fused filter without its table");
    if constexpr (AX == 0) {
        return launch_x<K, SW, false>(ax, cm, sw, gy, s);
    } else {
        const int TL = block_lines<K, AX, SW>(ax.P, ax.ftl);
        return launch_yz<K, AX, SW, false>(ax, cm, sw, TL, true, direct_lds<SW>(ax.P, TL, false), gy, s);
    }
}

template <int AX, class SW>
static int dispatch(const AxisDesc& ax, const SweepCommon& cm, const SW& sw, hipStream_t s) {
    if constexpr (AX == 0) {
        if constexpr (SW::kGcbc)
            if (ax.gcbc) return launch_sweep<8, AX, SW, true>(ax, cm, sw, s);
        return launch_sweep<8, AX, SW, false>(ax, cm, sw, s);
    } else {
        if constexpr (SW::kGcbc) {
            if (ax.gcbc && ax.K == 8) return launch_sweep<8, AX, SW, true>(ax, cm, sw, s);
            if (ax.gcbc) return launch_sweep<16, AX, SW, true>(ax, cm, sw, s);
        }
        if (ax.K == 8) return launch_sweep<8, AX, SW, false>(ax, cm, sw, s);
        return launch_sweep<16, AX, SW, false>(ax, cm, sw, s);
    }
}

// ---------------------------------------------------------------------------
// host orchestration
// ---------------------------------------------------------------------------
// the solver's FP64 buffers of the viscous intermediates hold FP32 fields of
// the same point count when the intermediates are stored in FP32
template <class TS>
inline TS* store_of(double* p) { return reinterpret_cast<TS*>(p); }

template <template <int, bool> class F, int AX, bool CLOSE>
static F<AX, CLOSE> make_s1(const cs_solver* sv, const double* q) {
    typedef typename F<AX, CLOSE>::Store TS;
    F<AX, CLOSE> a{};
    const long lmx = sv->g.lmx;
    fields(q, lmx, a.q);
    const int* axes = kS1Axes[sv->order];
    if constexpr (!CLOSE) {
        fields(store_of<TS>(AX == axes[0] ? sv->ga : sv->gb), lmx, a.gout);
    } else {
        for (int a2 = 0; a2 < 3; a2++) {
            const TS* g = a2 == axes[0] ? store_of<TS>(sv->ga) : (a2 == axes[1] ? store_of<TS>(sv->gb) : nullptr);
            fields(g, lmx, a.gin[a2]);
        }
        fields(store_of<TS>(sv->tau), lmx, a.tau);
        fields(store_of<TS>(sv->hf), lmx, a.hf);
    }
    a.ph = phys_of(sv);
    if constexpr (F<AX, CLOSE>::kCurv) a.mt = sv->met;
    return a;
}

template <template <int, int, bool> class F, int AX, int MODE, bool V>
static F<AX, MODE, V> make_s2(const cs_solver* sv, const double* q, const double* din, double* dout,
                               const double* q0, int div) {
    typedef typename F<AX, MODE, V>::Store TS;
    F<AX, MODE, V> a{};
    const long lmx = sv->g.lmx;
    fields(q, lmx, a.q);
    if (V) {
        const int t0 = AX == 0 ? 0 : (AX == 1 ? 3 : 5);
        const int t1 = AX == 0 ? 3 : (AX == 1 ? 1 : 4);
        const int t2 = AX == 0 ? 5 : (AX == 1 ? 4 : 2);
        const TS* tau = store_of<TS>(sv->tau);
        a.tr[0] = tau + (long)t0 * lmx;
        a.tr[1] = tau + (long)t1 * lmx;
        a.tr[2] = tau + (long)t2 * lmx;
        if constexpr (F<AX, MODE, V>::kHeat)
            a.hx = store_of<TS>(AX == kS1Axes[sv->order][0] ? sv->ga : sv->gb) + 3 * lmx;
        else
            a.hx = store_of<TS>(sv->hf) + (long)AX * lmx;
        if constexpr (F<AX, MODE, V>::kCurv) {
            fields(tau, lmx, a.tau6);
            fields((const TS*)store_of<TS>(sv->hf), lmx, a.h3);
        }
    }
    if constexpr (F<AX, MODE, V>::kCurv) a.mt = sv->met;
    fields(din, lmx, a.din);
    fields(dout, lmx, a.dout);
    fields(q0, lmx, a.q0);
    a.dtp = sv->dt;
    a.div = div;
    a.ph = phys_of(sv);
    a.nface = sv->g.face_size(AX);
    a.rec = sv->rec ? sv->rec + face_offset(sv->g, AX) : nullptr;
    a.lxi = sv->g.lxi;
    a.plane = (long)sv->g.lxi * sv->g.let;
    return a;
}

// sweep `pos` of one RHS (0..2 = S1 sweeps, 3..5 = S2 sweeps, in the
// solver's order); the last S2 sweep writes the RHS to `out`, or, when q0 is
// given, the RK stage q0 - dt/div*J*RHS
template <bool V, template <int, int, bool> class F = S2>
static int s2_sweep(cs_solver* sv, int k, const SweepCommon& cm, const double* q, double* out, const double* q0,
                    int div, hipStream_t s) {
    const int ax = kS2Axes[sv->order][k];
    if (k == 0) {
        if (ax == 0) return dispatch<0>(sv->rax[0], cm, make_s2<F, 0, 0, V>(sv, q, nullptr, sv->dpart, nullptr, 0), s);
        return dispatch<2>(sv->rax[2], cm, make_s2<F, 2, 0, V>(sv, q, nullptr, sv->dpart, nullptr, 0), s);
    }
    if (k == 1) return dispatch<1>(sv->rax[1], cm, make_s2<F, 1, 1, V>(sv, q, sv->dpart, sv->dpart, nullptr, 0), s);
    if (ax == 2) {
        if (q0) return dispatch<2>(sv->rax[2], cm, make_s2<F, 2, 3, V>(sv, q, sv->dpart, out, q0, div), s);
        return dispatch<2>(sv->rax[2], cm, make_s2<F, 2, 2, V>(sv, q, sv->dpart, out, nullptr, 0), s);
    }
    if (q0) return dispatch<0>(sv->rax[0], cm, make_s2<F, 0, 3, V>(sv, q, sv->dpart, out, q0, div), s);
    return dispatch<0>(sv->rax[0], cm, make_s2<F, 0, 2, V>(sv, q, sv->dpart, out, nullptr, 0), s);
}

// the gradient functor that also reduces the time step, per storage type
template <template <int, bool> class F>
struct DtOf {
    static constexpr bool kOk = false;
    template <int A, bool C>
    using type = F<A, C>;
};
template <>
struct DtOf<S1> {
    static constexpr bool kOk = true;
    template <int A, bool C>
    using type = S1D<A, C>;
};
template <>
struct DtOf<S1F> {
    static constexpr bool kOk = true;
    template <int A, bool C>
    using type = S1FD<A, C>;
};
template <>
struct DtOf<S1C> {
    static constexpr bool kOk = true;
    template <int A, bool C>
    using type = S1CD<A, C>;
};
template <>
struct DtOf<S1CF> {
    static constexpr bool kOk = true;
    template <int A, bool C>
    using type = S1CFD<A, C>;
};

template <template <int, bool> class F = S1>
static int s1_sweep(cs_solver* sv, int k, const SweepCommon& cm, const double* q, hipStream_t s) {
    if (sv->order == 0) {
        if (k == 0) return dispatch<0>(sv->rax[0], cm, make_s1<F, 0, false>(sv, q), s);
        if (k == 1) return dispatch<1>(sv->rax[1], cm, make_s1<F, 1, false>(sv, q), s);
        return dispatch<2>(sv->rax[2], cm, make_s1<F, 2, true>(sv, q), s);
    }
    // the sweep of an RK4 step's first stage that reduces the time step
    // (dt_fold = its position + 1): the first with constant metrics, the
    // closing x sweep with per-point metrics
    if (k == 0) {
        if constexpr (DtOf<F>::kOk && !F<1, false>::kCurv) {
            if (sv->dt_fold == 1) {
                auto f = make_s1<DtOf<F>::template type, 1, false>(sv, q);
                f.dtpart = sv->dtpart;
                return dispatch<1>(sv->rax[1], cm, f, s);
            }
        }
        return dispatch<1>(sv->rax[1], cm, make_s1<F, 1, false>(sv, q), s);
    }
    if (k == 1) return dispatch<2>(sv->rax[2], cm, make_s1<F, 2, false>(sv, q), s);
    if constexpr (DtOf<F>::kOk && F<0, true>::kCurv) {
        if (sv->dt_fold == 3) {
            auto f = make_s1<DtOf<F>::template type, 0, true>(sv, q);
            f.dtpart = sv->dtpart;
            return dispatch<0>(sv->rax[0], cm, f, s);
        }
    }
    return dispatch<0>(sv->rax[0], cm, make_s1<F, 0, true>(sv, q), s);
}

}  // namespace fused
}  // namespace cs
