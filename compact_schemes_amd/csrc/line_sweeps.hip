// line_sweeps.hip -- the derivative and the filter of single fields on the
// kernels of the fused sweeps (fused_kernels.hpp): what cs_deriv, cs_filter,
// the per-operator right-hand side and the batch launch for FP64 operators
// whose line splits into chunks at most one row short, seam sums (if any)
// formed from the line itself.  Everything else -- received seam sums, mixed
// precision, lines that do not split so or are longer -- runs line_solver.hip.
#include "fused_kernels.hpp"

namespace cs {
namespace fused {

// One field from `in` to `out` (which may be the same: every row of a line is
// loaded before one is stored); grid.y runs fields fstride (ostride) apart.
template <bool FILTER>
struct LineSweep {
    static constexpr int NF = 1;
    static constexpr bool kBlocks = false;
    static constexpr int kBytes = 16;
    static constexpr bool kGcbc = false;
    static constexpr int kStash = 0;
    static constexpr int kH = FILTER ? 5 : 2;
    static constexpr int kWpe = 4;
    static constexpr int kWpe16 = 4;
    static constexpr bool kFilter = FILTER;
    static constexpr bool kAdds = false;
    static constexpr bool kEnds = !FILTER;
    const double* in;
    double* out;
    long fstride, ostride;
    double* drva;     // [2 face][5 var][nface] from the first field's variable on, or null
    long nface;
    struct Raw { double q; };
    template <bool NT>
    __device__ __forceinline__ void load(uoff bo, Raw& w) const { w.q = ldg<NT>(in + (long)blockIdx.y * fstride, bo); }
    __device__ __forceinline__ void eval(const Raw& w, double* v) const { v[0] = w.q; }
    template <bool NT>
    __device__ __forceinline__ void store(uoff bo, const double* d) const { stg<NT>(out + (long)blockIdx.y * ostride, bo, d[0]); }
    // boundary derivatives for the characteristic BCs
    __device__ __forceinline__ void end_value(int face, long line, double v) const {
        if (drva) drva[((long)face * kNV + (long)blockIdx.y) * nface + line] = v;
    }
};
typedef LineSweep<false> LineDeriv;
typedef LineSweep<true> LineFilter;

// lines per workgroup of y/z lines: 64 (one chunk a wave, scalar table loads,
// 512-byte rows) up to 16 chunks, else 16
static int sweep_lines(int axis, int P) { return axis == 0 ? 64 / P : (P <= 16 ? 64 : 16); }

static AxisDesc axis_of(const LineArgs& a, int K, bool filter) {
    AxisDesc d{};
    d.tab = d.ftab = a.chunks;
    d.N = a.N;
    d.P = a.P;
    d.K = K;
    d.nlines = a.nlines;
    d.st = a.st;
    d.seam = filter ? a.cyclic : a.seam0;
    return d;
}

static SweepCommon common_of(const LineArgs& a) {
    SweepCommon c{};
    c.lxi = a.lxi;
    c.plane = a.plane;
    c.pb = a.pb;
    return c;
}

template <bool FILTER>
static LineSweep<FILTER> sweep_of(const LineArgs& a) {
    LineSweep<FILTER> w{};
    w.in = a.in;
    w.out = a.out;
    w.fstride = a.fstride;
    w.ostride = a.ostride;
    w.nface = a.nlines;
    w.drva = a.drva ? a.drva + (long)a.var * a.nlines : nullptr;
    return w;
}

template <int K, int AX, bool FILTER>
static int launch_one(const LineArgs& a, hipStream_t s) {
    typedef LineSweep<FILTER> SW;
    const AxisDesc ax = axis_of(a, K, FILTER);
    const SweepCommon cm = common_of(a);
    const SW sw = sweep_of<FILTER>(a);
    const unsigned gy = a.nfields > 1 ? (unsigned)a.nfields : 1u;
    if constexpr (AX == 0) {
        return launch_x<K, SW, false>(ax, cm, sw, gy, s);
    } else {
        const int TL = sweep_lines(AX, ax.P);
        const bool exact = ax.N == ax.P * K, nt = streams<SW>(ax, cm, gy);
        const void* k = TL == 64 ? (exact ? (nt ? (const void*)direct_kernel<K, AX, 64, SW, false, true, true>
                                                : (const void*)direct_kernel<K, AX, 64, SW, false, true, false>)
                                          : (nt ? (const void*)direct_kernel<K, AX, 64, SW, false, false, true>
                                                : (const void*)direct_kernel<K, AX, 64, SW, false, false, false>))
                                 : (nt ? (const void*)direct_kernel<K, AX, 16, SW, false, false, true>
                                       : (const void*)direct_kernel<K, AX, 16, SW, false, false, false>);
        const dim3 grid((unsigned)((ax.nlines + TL - 1) / TL), gy);
        return launch(k, grid, dim3(TL * ax.P), direct_lds<SW>(ax.P, TL, ax.seam),
                      with_runs(ax, grid.x, true, (AX == 1 ? 128 : 1024) / TL), cm, sw, s);
    }
}

template <int K, bool FILTER>
static int launch_axis(int axis, const LineArgs& a, hipStream_t s) {
    if (axis == 0) return launch_one<K, 0, FILTER>(a, s);
    if (axis == 1) return launch_one<K, 1, FILTER>(a, s);
    return launch_one<K, 2, FILTER>(a, s);
}

// ---------------------------------------------------------------------------
// batched: the same kernels, items dealt over the grid (any chunk lengths in
// one class, so the bits are those of the single launches)
// ---------------------------------------------------------------------------
template <int K, bool FILTER>
static const void* batch_kernel(int axis, int P) {
    typedef LineSweep<FILTER> SW;
    typedef BatchItems<SW> B;
    if (axis == 0) return (const void*)xt_kernel<K, SW, false, false, false, B>;
    if (sweep_lines(axis, P) == 64)
        return axis == 1 ? (const void*)direct_kernel<K, 1, 64, SW, false, false, false, B>
                         : (const void*)direct_kernel<K, 2, 64, SW, false, false, false, B>;
    return axis == 1 ? (const void*)direct_kernel<K, 1, 16, SW, false, false, false, B>
                     : (const void*)direct_kernel<K, 2, 16, SW, false, false, false, B>;
}

static const void* batch_kernel(int op, int K, int axis, int P) {
    if (op == OP_FILTER) return K == 8 ? batch_kernel<8, true>(axis, P) : batch_kernel<16, true>(axis, P);
    return K == 8 ? batch_kernel<8, false>(axis, P) : batch_kernel<16, false>(axis, P);
}

template <bool FILTER>
static void pack(const LineArgs& a, int K, unsigned char* dst) {
    const BatchOp<LineSweep<FILTER>> o{axis_of(a, K, FILTER), common_of(a), sweep_of<FILTER>(a)};
    __builtin_memcpy(dst, &o, sizeof o);
}

template <bool FILTER>
static int launch_items(const void* k, dim3 grid, dim3 block, size_t lds, const void* ops, const int2* items, int n,
                        hipStream_t s) {
    typedef LineSweep<FILTER> SW;
    const BatchItems<SW> b{static_cast<const BatchOp<SW>*>(ops), items, n};
    return launch(k, grid, block, lds, AxisDesc{}, SweepCommon{}, SW{}, s, b);
}

}  // namespace fused

using namespace fused;

// Whether this operator runs the sweep kernels (a.P chunks of K points)
bool line_sweep_ok(int op, int axis, int K, const LineArgs& a) {
    if (!a.chunks || a.mixed || a.recv || (op != OP_DERIV && op != OP_FILTER) || (K != 8 && K != 16)) return false;
    if (op == OP_DERIV && a.seam0 != a.seam1) return false;
    if ((long)a.N * a.nlines > (1L << 29)) return false;             // 32-bit byte offsets
    return axis == 0 ? a.P <= 64 : a.P <= fused::kMaxP;
}

int launch_line_sweep(int op, int axis, int K, const LineArgs& a, hipStream_t s) {
    if (op == OP_FILTER) return K == 8 ? launch_axis<8, true>(axis, a, s) : launch_axis<16, true>(axis, a, s);
    return K == 8 ? launch_axis<8, false>(axis, a, s) : launch_axis<16, false>(axis, a, s);
}

int batch_sweep_lines(int axis, int P) { return sweep_lines(axis, P); }
int batch_sweep_threads(int axis, int P) { return axis == 0 ? 64 : sweep_lines(axis, P) * P; }
size_t batch_sweep_bytes() { return sizeof(BatchOp<LineDeriv>); }

size_t batch_sweep_lds(int op, int K, int axis, int P) {
    if (axis == 0) return K == 8 ? xt_lds<8, LineDeriv>(P) : xt_lds<16, LineDeriv>(P);
    const int TL = sweep_lines(axis, P);
    return op == OP_FILTER ? direct_lds<LineFilter>(P, TL, true) : direct_lds<LineDeriv>(P, TL, true);
}

void batch_sweep_pack(int op, int K, const LineArgs& a, unsigned char* dst) {
    static_assert(sizeof(BatchOp<LineDeriv>) == sizeof(BatchOp<LineFilter>), "one record size");
    if (op == OP_FILTER) pack<true>(a, K, dst);
    else pack<false>(a, K, dst);
}

int batch_sweep_blocks_per_cu(int op, int K, int axis, int P, size_t lds, int* nb) {
    const void* k = batch_kernel(op, K, axis, P);
    if (lds > 64 * 1024) CS_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int n = 0;
    CS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, batch_sweep_threads(axis, P), lds));
    *nb = n < 1 ? 1 : n;
    return CS_OK;
}

int launch_batch_sweeps(int op, int K, int axis, int P, const void* ops, const int2* items, int nitems, int grid,
                        size_t lds, hipStream_t s) {
    if (nitems <= 0) return CS_OK;
    const void* k = batch_kernel(op, K, axis, P);
    const dim3 g((unsigned)grid), b((unsigned)batch_sweep_threads(axis, P));
    return op == OP_FILTER ? launch_items<true>(k, g, b, lds, ops, items, nitems, s)
                           : launch_items<false>(k, g, b, lds, ops, items, nitems, s);
}

}  // namespace cs
