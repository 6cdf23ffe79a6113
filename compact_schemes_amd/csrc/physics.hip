// physics.hip -- pointwise kernels of the compressible right-hand side.
//
// Each kernel computes what the reference kernel named in its comment
// computes (src/cuda/kernels/physics.hpp of EnricoDeg/compact_schemes) on the
// same SoA layout; corrections of reference defects are named where applied.
// All are one-point-per-thread streaming kernels: HBM-bound, 256 threads.
#include "physics_kernels.hpp"

#include <cmath>
#include <mutex>
#include <string>

namespace cs {

constexpr int kBlock = 256;

// with the streaming hint where NT
template <bool NT>
__device__ __forceinline__ double ld(const double* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT>
__device__ __forceinline__ void st(double* p, double v) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}
// The hint pays where a kernel passes over more than the last-level cache
// holds (160x128x96, 42 fields: fluxes_pre 120 -> 108 us, visc 108 -> 91);
// below, the next kernel finds there what this one wrote (96x80x64: the
// step 798 us without the hint there, 808 with it).
static bool streams(int nfields, long lmx) { return 8.0 * nfields * (double)lmx > 256.0 * (1 << 20); }

static dim3 grid_for(long n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

// primitive variables (absent upstream): de0 = 1/rho, de1..3 = u, v, w,
// de4 = c^2 = gam p / rho, p = (gam-1)(E - rho |u|^2 / 2)
__global__ void __launch_bounds__(kBlock) primitives_kernel(const double* qa, double* de, double* p, long lmx) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    double q[5];
    load_q(qa, t, lmx, q);
    Prim w = primitive(q);
    de[t] = w.rhoi;
    de[t + lmx] = w.u;
    de[t + 2 * lmx] = w.v;
    de[t + 3 * lmx] = w.w;
    de[t + 4 * lmx] = w.c2;
    p[t] = w.p;
}

// calc_fluxes_pre_compute_kernel, src/cuda/kernels/physics.hpp:42-193
// (D21 intended: stress/heat are not read when Visc is false; the E + p it
// leaves in de is overwritten by the flux divergence and not written here).
template <bool Visc, bool NT>
__global__ void __launch_bounds__(kBlock) fluxes_pre_kernel(double* buffer, const double* qa, const double* pr,
                                                            const double* de, const double* xim, const double* etm,
                                                            const double* zem, const double* stress,
                                                            const double* heat, cs_point umf, long lmx) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    double q[5], u[3], mt[3][3], tau[6] = {0, 0, 0, 0, 0, 0}, hf[3] = {0, 0, 0};
    for (int v = 0; v < 5; v++) q[v] = ld<NT>(qa + t + v * lmx);
    for (int d = 0; d < 3; d++) u[d] = ld<NT>(de + t + (d + 1) * lmx);
    for (int d = 0; d < 3; d++) {
        mt[0][d] = ld<NT>(xim + t + d * lmx);
        mt[1][d] = ld<NT>(etm + t + d * lmx);
        mt[2][d] = ld<NT>(zem + t + d * lmx);
    }
    if (Visc) {
        for (int k = 0; k < 6; k++) tau[k] = ld<NT>(stress + t + k * lmx);
        for (int k = 0; k < 3; k++) hf[k] = ld<NT>(heat + t + k * lmx);
    }
    double F[5][3];
    flux_all<Visc>(q, ld<NT>(pr + t), u, mt, tau, hf, umf, F);
    for (int m = 0; m < 5; m++)
        for (int j = 0; j < 3; j++) st<NT>(buffer + t + (long)(3 * m + j) * lmx, F[m][j]);
}

// calc_fluxes_post_compute_kernel<m>, src/cuda/kernels/physics.hpp:195-209,
// for all five variables
template <bool NT>
__global__ void __launch_bounds__(kBlock) fluxes_post_kernel(double* de, const double* bd, long lmx) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    double d[kNV][3];
    for (int m = 0; m < kNV; m++)
        for (int j = 0; j < 3; j++) d[m][j] = ld<NT>(bd + t + (long)(3 * m + j) * lmx);
    for (int m = 0; m < kNV; m++) st<NT>(de + t + (long)m * lmx, d[m][0] + d[m][1] + d[m][2]);
}

// calc_viscous_shear_stress_post_compute_kernel<m> (m = 1..4) and
// calc_viscous_shear_stress_final_kernel, src/cuda/kernels/physics.hpp:228-333,
// D8 intended (reads the derivatives): the physical gradients of u, v, w, c^2
// from the index-space ones bd[m][3] and the metrics, then stress and heat
// flux.  The reference passes the twelve gradients through the stress and
// heat arrays (five kernels, 84 fields read or written); in registers the
// 26 reads and 11 writes are left, and they are the bound (160x128x96: five
// kernels 229 us, this one 91 = 6.4 TB/s).
template <bool NT>
__global__ void __launch_bounds__(kBlock) visc_kernel(double* de, const double* ssk, const double* yaco,
                                                      const double* bd, const double* xim, const double* etm,
                                                      const double* zem, double* stress, double* heat, long lmx) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    double mt[3][3], f[4][3], u[3];
    for (int d = 0; d < 3; d++) {
        mt[0][d] = ld<NT>(xim + t + d * lmx);
        mt[1][d] = ld<NT>(etm + t + d * lmx);
        mt[2][d] = ld<NT>(zem + t + d * lmx);
        u[d] = ld<NT>(de + t + (d + 1) * lmx);
    }
    for (int m = 0; m < 4; m++)
        for (int j = 0; j < 3; j++) f[m][j] = ld<NT>(bd + t + (long)(3 * (m + 1) + j) * lmx);
    const double mu = ld<NT>(ssk + t), J = ld<NT>(yaco + t);
    double g[12];   // (u_x, u_y, u_z, v_x, v_y, v_z, w_x, w_y, w_z, c2_x, c2_y, c2_z)
    for (int m = 0; m < 4; m++)
        for (int d = 0; d < 3; d++) g[3 * m + d] = mt[0][d] * f[m][0] + mt[1][d] * f[m][1] + mt[2][d] * f[m][2];
    double tau[6], hf[3], d4;
    viscous_closure(mu, J, g, g + 9, u, tau, hf, &d4);
    st<NT>(de + t, mu);
    st<NT>(de + t + 4 * lmx, d4);
    for (int k = 0; k < 6; k++) st<NT>(stress + t + k * lmx, tau[k]);
    for (int k = 0; k < 3; k++) st<NT>(heat + t + k * lmx, hf[k]);
}

// calc_time_step_kernel, src/cuda/kernels/physics.hpp:335-427 (D9 intended:
// FP64 max, lanes past the end and the accumulators start at 0).  Stage 1
// writes one pair of partial maxima per block; stage 2 reduces them.
__global__ void __launch_bounds__(kBlock) time_step_kernel(const double* xim, const double* etm, const double* zem,
                                                           const double* de, const double* yaco, const double* ssk,
                                                           cs_point umf, double* part, long lmx) {
    __shared__ double s0[kBlock], s1[kBlock];
    double m0 = 0.0, m1 = 0.0;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < lmx; t += (long)gridDim.x * blockDim.x) {
        double rr1 = 0.0;
        for (int d = 0; d < 3; d++) rr1 += xim[t + d * lmx] * xim[t + d * lmx];
        for (int d = 0; d < 3; d++) rr1 += etm[t + d * lmx] * etm[t + d * lmx];
        for (int d = 0; d < 3; d++) rr1 += zem[t + d * lmx] * zem[t + d * lmx];
        double u = de[t + lmx] + umf.x, v = de[t + 2 * lmx] + umf.y, w = de[t + 3 * lmx] + umf.z;
        double rr2 = fabs(xim[t] * u + xim[t + lmx] * v + xim[t + 2 * lmx] * w) +
                     fabs(etm[t] * u + etm[t + lmx] * v + etm[t + 2 * lmx] * w) +
                     fabs(zem[t] * u + zem[t + lmx] * v + zem[t + 2 * lmx] * w);
        double ssi = fabs(yaco[t]);
        m0 = fmax(m0, (sqrt(de[t + 4 * lmx] * rr1) + rr2) * ssi);
        m1 = fmax(m1, de[t] * ssk[t] * rr1 * ssi * ssi);
    }
    s0[threadIdx.x] = m0;
    s1[threadIdx.x] = m1;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s0[threadIdx.x] = fmax(s0[threadIdx.x], s0[threadIdx.x + w]);
            s1[threadIdx.x] = fmax(s1[threadIdx.x], s1[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = s0[0]; part[2 * blockIdx.x + 1] = s1[0]; }
}

// out3 (may be null): also writes dte = min(cfl / max0, 0.5 / max1) and the
// two maxima, so a caller that does not synchronise gets the time step on the device
__global__ void __launch_bounds__(kBlock) max_pairs_kernel(double* part, int n, double cfl, double* out3) {
    __shared__ double s0[kBlock], s1[kBlock];
    double m0 = 0.0, m1 = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) { m0 = fmax(m0, part[2 * i]); m1 = fmax(m1, part[2 * i + 1]); }
    s0[threadIdx.x] = m0;
    s1[threadIdx.x] = m1;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s0[threadIdx.x] = fmax(s0[threadIdx.x], s0[threadIdx.x + w]);
            s1[threadIdx.x] = fmax(s1[threadIdx.x], s1[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * n] = s0[0];
        part[2 * n + 1] = s1[0];
        if (out3) {
            out3[0] = fmin(cfl / s0[0], 0.5 / s1[0]);
            out3[1] = s0[0];
            out3[2] = s1[0];
        }
    }
}

// RK stage update (absent upstream): q = q0 - dtk * yaco * de
__global__ void __launch_bounds__(kBlock) rk_stage_kernel(double* q, const double* q0, const double* de,
                                                          const double* yaco, double dtk, long lmx) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    double f = dtk * yaco[t];
    for (int v = 0; v < 5; v++) q[t + v * lmx] = q0[t + v * lmx] - f * de[t + v * lmx];
}

// initial state: uniform flow at rest in the frame (stored velocity 0),
// rho0 = 1, p0 = 1/gam, and a Gaussian pressure pulse with rho' = p' (c0 = 1)
__global__ void __launch_bounds__(kBlock) init_pulse_kernel(double* qa, int lxi, int let, long lmx, cs_point cen,
                                                            double amp, double width) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    const long plane = (long)lxi * let;
    const double z = (double)(t / plane), y = (double)((t % plane) / lxi), x = (double)(t % lxi);
    const double r2 = (x - cen.x) * (x - cen.x) + (y - cen.y) * (y - cen.y) + (z - cen.z) * (z - cen.z);
    const double pp = amp * exp(-M_LN2 * r2 / (width * width));
    qa[t] = 1.0 + pp;
    qa[t + lmx] = 0.0;
    qa[t + 2 * lmx] = 0.0;
    qa[t + 3 * lmx] = 0.0;
    qa[t + 4 * lmx] = (kHam + pp) / kGamm1;
}

// sbcc: 1 on the boundary points of the subdomain, 0 inside
__global__ void __launch_bounds__(kBlock) boundary_weights_kernel(double* sbcc, int lxi, int let, int lze, long lmx) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lmx) return;
    const long plane = (long)lxi * let;
    const long z = t / plane, y = (t % plane) / lxi, x = t % lxi;
    const bool on = x == 0 || x == lxi - 1 || y == 0 || y == let - 1 || z == 0 || z == lze - 1;
    sbcc[t] = on ? 1.0 : 0.0;
}

// fill_gpu_buffer_kernel<Axis>, src/cuda/kernels/numerics_pc.hpp:42-122: for
// every line of the face, the two pbco-weighted 8-point sums from the face
// inward (istart/increment of numerics_pc.hpp:275-280).
__global__ void __launch_bounds__(kBlock) fill_kernel(const double* in, double* send, const double* pbco, int axis,
                                                      int face, int N, long nlines, int lxi, long plane, long st) {
    long f = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nlines) return;
    long b = line_base(axis, f, lxi, plane);
    int istart = face * (N - 1), inc = 1 - 2 * face;
    double v0 = 0.0, v1 = 0.0;
    for (int i = 0; i < kLmd; i++) {
        double x = in[b + (long)(istart + inc * i) * st];
        v0 += pbco[i] * x;
        v1 += pbco[kLmd + i] * x;
    }
    send[f] = v0;
    send[nlines + f] = v1;
}

// ---------------------------------------------------------------------------
int launch_primitives(const double* qa, double* de, double* p, long lmx, hipStream_t s) {
    hipLaunchKernelGGL(primitives_kernel, grid_for(lmx), dim3(kBlock), 0, s, qa, de, p, lmx);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_fluxes_pre(bool visc, double* buffer, const double* qa, const double* p, const double* de,
                      const double* xim, const double* etm, const double* zem, const double* stress,
                      const double* heat, cs_point umf, long lmx, hipStream_t s) {
    const bool nt = streams(visc ? 42 : 33, lmx);
    auto k = visc ? (nt ? fluxes_pre_kernel<true, true> : fluxes_pre_kernel<true, false>)
                  : (nt ? fluxes_pre_kernel<false, true> : fluxes_pre_kernel<false, false>);
    hipLaunchKernelGGL(k, grid_for(lmx), dim3(kBlock), 0, s, buffer, qa, p, de, xim, etm, zem, stress, heat, umf, lmx);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_fluxes_post(double* de, const double* bd, long lmx, hipStream_t s) {
    auto k = streams(20, lmx) ? fluxes_post_kernel<true> : fluxes_post_kernel<false>;
    hipLaunchKernelGGL(k, grid_for(lmx), dim3(kBlock), 0, s, de, bd, lmx);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_visc(double* de, const double* ssk, const double* yaco, const double* bd, const double* xim,
                const double* etm, const double* zem, double* stress, double* heat, long lmx, hipStream_t s) {
    auto k = streams(37, lmx) ? visc_kernel<true> : visc_kernel<false>;
    hipLaunchKernelGGL(k, grid_for(lmx), dim3(kBlock), 0, s, de, ssk, yaco, bd, xim, etm, zem, stress, heat,
                       lmx);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int time_step_blocks(long lmx) {
    long b = (lmx + kBlock - 1) / kBlock;
    return (int)(b < 2048 ? b : 2048);
}

int launch_time_step(const double* xim, const double* etm, const double* zem, const double* de, const double* yaco,
                     const double* ssk, cs_point umf, double* part, int nblocks, long lmx, hipStream_t s) {
    hipLaunchKernelGGL(time_step_kernel, dim3(nblocks), dim3(kBlock), 0, s, xim, etm, zem, de, yaco, ssk, umf, part,
                       lmx);
    CS_HIP(hipGetLastError());
    hipLaunchKernelGGL(max_pairs_kernel, dim3(1), dim3(kBlock), 0, s, part, nblocks, 0.0, (double*)nullptr);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_rk_stage(double* q, const double* q0, const double* de, const double* yaco, double dtk, long lmx,
                    hipStream_t s) {
    hipLaunchKernelGGL(rk_stage_kernel, grid_for(lmx), dim3(kBlock), 0, s, q, q0, de, yaco, dtk, lmx);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_fill(const double* in, double* send, const double* pbco, int axis, int face, int N, long nlines, int lxi,
                long plane, long st, hipStream_t s) {
    hipLaunchKernelGGL(fill_kernel, grid_for(nlines), dim3(kBlock), 0, s, in, send, pbco, axis, face, N, nlines, lxi,
                       plane, st);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_init_pulse(const cs_dims* d, cs_point cen, double amp, double width, double* qa, hipStream_t s) {
    const long lmx = (long)d->lxi * d->let * d->lze;
    hipLaunchKernelGGL(init_pulse_kernel, grid_for(lmx), dim3(kBlock), 0, s, qa, d->lxi, d->let, lmx, cen, amp, width);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

int launch_boundary_weights(const cs_dims* d, double* sbcc, hipStream_t s) {
    const long lmx = (long)d->lxi * d->let * d->lze;
    hipLaunchKernelGGL(boundary_weights_kernel, grid_for(lmx), dim3(kBlock), 0, s, sbcc, d->lxi, d->let, d->lze, lmx);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

// ---------------------------------------------------------------------------
// allocation-free time step
// ---------------------------------------------------------------------------
// Scratch of cs_calc_time_step_noalloc: one pair of partial maxima per block
// of time_step_kernel and the reduced pair (kTsMaxBlocks pairs + 1, 32.8 KB).
// Each GPU holds its own copy from the library's load until the process ends,
// shared by every call on that GPU.  Nothing in it needs clearing: every block
// writes its pair before max_pairs_kernel reads it.  In host code the name is
// a stand-in, never a device address: kernels get the per-device pointer
// from hipGetSymbolAddress.
constexpr int kTsMaxBlocks = 2048;
static __device__ __align__(256) double scratch[2 * kTsMaxBlocks + 2];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch[kMaxDevices] = {};
}  // namespace

// device address of `scratch` on the current device, looked up on the first
// call on each device
static int scratch_on_device(double** out) {
    int dev = 0;
    CS_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(CS_ERR_UNSUPPORTED, "device ordinal above 63");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        CS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(CS_ERR_HIP, "hipGetSymbolAddress returned a null address for the time-step scratch");
        g_scratch[dev] = static_cast<double*>(p);
    }
    *out = g_scratch[dev];
    return CS_OK;
}

}  // namespace cs

using namespace cs;

extern "C" int cs_calc_time_step_noalloc(const cs_dims* dims, cs_point umf, const double* xim, const double* etm,
                                         const double* zem, const double* de, const double* yaco, const double* ssk,
                                         double cfl, double* out3, cs_stream stream) {
    if (!dims || !out3) return fail(CS_ERR_ARG, "null argument");
    if (!xim || !etm || !zem || !de || !yaco || !ssk) return fail(CS_ERR_ARG, "null field pointer");
    if (dims->lxi < 1 || dims->let < 1 || dims->lze < 1) return fail(CS_ERR_SHAPE, "grid dimensions must be positive");
    const long lmx = (long)dims->lxi * dims->let * dims->lze;
    const int nblocks = time_step_blocks(lmx);
    if (nblocks > kTsMaxBlocks)
        return fail(CS_ERR_SHAPE, "time-step reduction needs " + std::to_string(nblocks) +
                                      " partial pairs; the static scratch holds " + std::to_string(kTsMaxBlocks));
    double* part = nullptr;
    int rc = scratch_on_device(&part);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(time_step_kernel, dim3(nblocks), dim3(kBlock), 0, s, xim, etm, zem, de, yaco, ssk, umf, part,
                       lmx);
    CS_HIP(hipGetLastError());
    hipLaunchKernelGGL(max_pairs_kernel, dim3(1), dim3(kBlock), 0, s, part, nblocks, cfl, out3);
    CS_HIP(hipGetLastError());
    return CS_OK;
}

extern "C" int cs_init_pulse(const cs_dims* dims, cs_point center, double amp, double width, double* qa,
                             cs_stream stream) {
    if (!dims || !qa) return fail(CS_ERR_ARG, "null argument");
    if (dims->lxi < 1 || dims->let < 1 || dims->lze < 1) return fail(CS_ERR_SHAPE, "grid dimensions must be positive");
    if (!(width > 0.0) || !std::isfinite(amp)) return fail(CS_ERR_ARG, "pulse width must be > 0 and amp finite");
    return launch_init_pulse(dims, center, amp, width, qa, (hipStream_t)stream);
}

extern "C" int cs_boundary_weights(const cs_dims* dims, double* sbcc, cs_stream stream) {
    if (!dims || !sbcc) return fail(CS_ERR_ARG, "null argument");
    if (dims->lxi < 1 || dims->let < 1 || dims->lze < 1) return fail(CS_ERR_SHAPE, "grid dimensions must be positive");
    return launch_boundary_weights(dims, sbcc, (hipStream_t)stream);
}
