// Multigrid transfer kernels for gfx950: K-tap restriction and
// interpolation (K = 2 nn = 2, 4, 6, 8), real and complex, periodic / zero /
// Bloch-phase boundaries.
//
// A 3-D transfer is the product of three 1-D transfers (z, then y, then x,
// the order of c/bmgs/restrict.cpp:153-155 and interpolate.cpp:86-97).
// Each pass is one kernel with one thread per output point; the boundary of
// the pass's axis is taken by index wrap, the other two axes are in range.
//
// 1-D semantics in interior-index form (derived from the reference's padded
// buffers, c/bmgs/restrict.cpp:18-63 and interpolate.cpp:10-46):
//   restrict:    out[i] = 1/2 (a[c] + sum_j w_j (a[c+j] + a[c-j])),
//                c = 2 i + off, j = 1, 3, .., K-1
//   interpolate: with p = (i + skip0) / 2, c = p + off:
//                even (i + skip0): out[i] = a[c]
//                odd:              out[i] = sum_j w_j (a[c-j] + a[c+1+j]),
//                j = 0 .. K/2-1
// The weights are exact dyadic rationals.
#include "transfer.h"

#include "batch.h"
#include "stencil_dev.h"

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>

#include <type_traits>

namespace gfd {

template <int K> struct W;
template <> struct W<2> {
    static constexpr double w[1] = {0.5};
};
template <> struct W<4> {
    static constexpr double w[2] = {0.5625, -0.0625};
};
template <> struct W<6> {
    static constexpr double w[3] = {0.58593750, -0.09765625, 0.01171875};
};
template <> struct W<8> {
    static constexpr double w[4] = {0.59814453125, -0.11962890625,
                                    0.02392578125, -0.00244140625};
};

template <typename T> struct XIsCplx { static constexpr bool value = false; };
template <> struct XIsCplx<double2> { static constexpr bool value = true; };
template <> struct XIsCplx<float2> { static constexpr bool value = true; };

// input value (possibly the wider FP64 type) as the compute type T
template <typename T, typename TI>
__device__ inline T narrow(TI v)
{
    if constexpr (std::is_same<T, TI>::value) {
        return v;
    } else if constexpr (XIsCplx<T>::value) {
        return T{(float)v.x, (float)v.y};
    } else {
        return (T)v;
    }
}

template <typename T>
struct XArgs {
    const T* in;
    T* out;
    T* out2;
    const T* base;
    int d[3];      // output dims of this pass
    int ilen;      // input length along the axis
    long istride;  // input stride along the axis
    long in_grid;  // input points per grid
    long out_grid; // output points per grid
    long total;
    int off, skip0;
    int periodic;
    double2 ph_hi, ph_lo;
    int negate;
    double alpha;
};

template <typename T>
__device__ inline T xload(const XArgs<T>& a, const T* __restrict__ g,
                          long pos, int j)
{
    if (j >= 0 && j < a.ilen) return g[pos + (long)j * a.istride];
    if (!a.periodic) return zero_of<T>();
    double2 f = make_double2(1.0, 0.0);
    bool first = true;
    while (j < 0) {
        j += a.ilen;
        f = first ? a.ph_lo : cmul(a.ph_lo, f);
        first = false;
    }
    while (j >= a.ilen) {
        j -= a.ilen;
        f = first ? a.ph_hi : cmul(a.ph_hi, f);
        first = false;
    }
    T v = g[pos + (long)j * a.istride];
    if constexpr (XIsCplx<T>::value) v = cmul(f, v);
    return v;
}

// One axis, one point per thread.
template <typename T, int AX, int K, bool INTERP, int EPI>
__global__ void __launch_bounds__(256) k_xfer1d(XArgs<T> a)
{
    typedef typename ScalarOf<T>::type S;
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= a.total) return;
    long b;
    int o0, o1, o2;
    flat_split(gid, a.total, a.out_grid, a.d[1], a.d[2], b, o0, o1, o2);
    // input position with the pass axis at 0
    const long pos = AX == 2   ? ((long)o0 * a.d[1] + o1) * a.ilen
                     : AX == 1 ? (long)o0 * a.ilen * a.d[2] + o2
                               : (long)o1 * a.d[2] + o2;
    const int i = AX == 2 ? o2 : AX == 1 ? o1 : o0;
    const T* __restrict__ g = a.in + b * a.in_grid;
    T v;
    if constexpr (!INTERP) {
        const int c = 2 * i + a.off;
        T acc = xload(a, g, pos, c);
#pragma unroll
        for (int m = 0; m < K / 2; m++) {
            const int j = 2 * m + 1;
            T pair = xload(a, g, pos, c + j) + xload(a, g, pos, c - j);
            acc = fmac(acc, (S)W<K>::w[m], pair);
        }
        v = (S)0.5 * acc;
    } else {
        const int q = i + a.skip0;
        const int c = (q >> 1) + a.off;
        if ((q & 1) == 0) {
            v = xload(a, g, pos, c);
        } else {
            T pair0 = xload(a, g, pos, c) + xload(a, g, pos, c + 1);
            T acc = (S)W<K>::w[0] * pair0;
#pragma unroll
            for (int m = 1; m < K / 2; m++) {
                T pair = xload(a, g, pos, c - m) + xload(a, g, pos, c + 1 + m);
                acc = fmac(acc, (S)W<K>::w[m], pair);
            }
            v = acc;
        }
    }
    if constexpr (EPI == XEPI_PLAIN) {
        a.out[gid] = v;
    } else if constexpr (EPI == XEPI_NEG) {
        a.out[gid] = -v;
    } else if constexpr (EPI == XEPI_SCALE2) {
        if (a.negate) v = -v;
        a.out[gid] = v;
        a.out2[gid] = (S)a.alpha * v;
    } else {
        a.out[gid] = a.base[gid] - v;
    }
}

// ------------------------------------------------------------ fused K = 2
// One thread per output point; the 3 x 3 x 3 fine neighbourhood
// (restriction) or the <= 8 coarse neighbours (interpolation) come through
// the caches.  Sums are associated z innermost, then y, then x, as the
// reference's pass order.

template <typename T, typename TI = T>
struct F3Args {
    const TI* in;
    T* out;
    T* out2;
    const T* base;
    int ni[3];      // input grid
    int no[3];      // output grid
    int off[3];     // interior index of the first centre per axis
    int skip0[3];
    int periodic[3];
    double2 ph[3][2];
    long in_grid, out_grid, total;
    int negate;
    double alpha;
};

// value of the input at (i0, i1, i2) with per-axis wrap / zero; the
// phase is applied at the input's precision, then the value is narrowed
template <typename T, typename TI>
__device__ inline T f3load(const F3Args<T, TI>& a, const TI* __restrict__ g,
                           int i0, int i1, int i2)
{
    int ii[3] = {i0, i1, i2};
    double2 f = make_double2(1.0, 0.0);
    bool phased = false;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        if (ii[c] >= 0 && ii[c] < a.ni[c]) continue;
        if (!a.periodic[c]) return zero_of<T>();
        while (ii[c] < 0) {
            ii[c] += a.ni[c];
            f = phased ? cmul(a.ph[c][1], f) : a.ph[c][1];
            phased = true;
        }
        while (ii[c] >= a.ni[c]) {
            ii[c] -= a.ni[c];
            f = phased ? cmul(a.ph[c][0], f) : a.ph[c][0];
            phased = true;
        }
    }
    TI v = g[((long)ii[0] * a.ni[1] + ii[1]) * a.ni[2] + ii[2]];
    if constexpr (XIsCplx<TI>::value)
        if (phased) v = apply_phase(v, f);
    return narrow<T, TI>(v);
}

template <typename T, int EPI, typename TI>
__device__ inline void f3store(const F3Args<T, TI>& a, long gid, T v)
{
    typedef typename ScalarOf<T>::type S;
    if constexpr (EPI == XEPI_PLAIN) {
        a.out[gid] = v;
    } else if constexpr (EPI == XEPI_NEG) {
        a.out[gid] = -v;
    } else if constexpr (EPI == XEPI_SCALE2) {
        if (a.negate) v = -v;
        a.out[gid] = v;
        a.out2[gid] = (S)a.alpha * v;
    } else {
        a.out[gid] = a.base[gid] - v;
    }
}

template <typename T, int EPI, typename TI>
__global__ void __launch_bounds__(256) k_restrict2(F3Args<T, TI> a)
{
    typedef typename ScalarOf<T>::type S;
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= a.total) return;
    long b;
    int o0, o1, o2;
    flat_split(gid, a.total, a.out_grid, a.no[1], a.no[2], b, o0, o1, o2);
    const int c0 = 2 * o0 + a.off[0], c1 = 2 * o1 + a.off[1],
              c2 = 2 * o2 + a.off[2];
    const TI* __restrict__ g = a.in + b * a.in_grid;
    T px[3];
#pragma unroll
    for (int dx = -1; dx <= 1; dx++) {
        T py[3];
#pragma unroll
        for (int dy = -1; dy <= 1; dy++) {
            // 1/2 (a0 + 1/2 (a1 + a-1)) along z
            const T zp = f3load(a, g, c0 + dx, c1 + dy, c2 + 1) +
                         f3load(a, g, c0 + dx, c1 + dy, c2 - 1);
            py[dy + 1] = (S)0.5 * fmac(f3load(a, g, c0 + dx, c1 + dy, c2),
                                       (S)0.5, zp);
        }
        px[dx + 1] = (S)0.5 * fmac(py[1], (S)0.5, py[2] + py[0]);
    }
    const T v = (S)0.5 * fmac(px[1], (S)0.5, px[2] + px[0]);
    f3store<T, EPI, TI>(a, gid, v);
}

// ------------------------------------------------- tiled K = 2 restriction
//
// A block stages the (2 CX + 1) x (2 CY + 1) x (2 cz + 1) fine points under
// its CX x CY x cz coarse ones in LDS, every load of the tile in flight at
// once (a wave per fine row, addresses uniform but for the lane), then forms
// each output from its 27 values.  One load latency and one barrier, where
// the marching kernel has one of each per fine plane and the
// one-point-per-thread kernel reads every fine point 3.4 times through L1
// with a stride of two.  A tile fits LDS three or four times per CU, and its
// rows are loaded in two rounds.  Measured, before (the faster of the two
// others) and with the tiles: 192^3 FP32 in the V-cycle 21.6 -> 16.0 us (read
// once 5); 8 complex grids of 128^3 84 -> 64 (50); 32 of 108x120x132 narrowed
// to FP32 283 -> 231 (160; 250 with five rounds of loads).  16 real grids of
// 96^3 stay with marching, 36 against 39: the kernel is timed per shape.
// Arrays of at least 2 GiB per grid (buffer offsets) stay with those.
template <typename T> struct RtTile {
    static constexpr int CX = sizeof(T) == 4 ? 4 : 2;
    static constexpr int CY = sizeof(T) == 16 ? 4 : 8;
};
constexpr int RT_CZ = 32;          // most coarse z points of a tile
constexpr int RT_P = 2 * RT_CZ + 1;

template <typename T, int EPI, typename TI>
__global__ void __launch_bounds__(256)
k_restrict_tile(F3Args<T, TI> a, int cz, int tiles_z, int tiles_y,
                int tiles_x, int nblocks)
{
    typedef typename ScalarOf<T>::type S;
    constexpr int CX = RtTile<T>::CX, CY = RtTile<T>::CY;
    constexpr int RX = 2 * CX + 1, RY = 2 * CY + 1, ROWS = RX * RY;
    constexpr bool CPLX = XIsCplx<TI>::value;
    __shared__ T E[ROWS * RT_P];
    int rem = xcd_remap(blockIdx.x, nblocks);
    const int zt = rem % tiles_z;
    rem /= tiles_z;
    const int yt = rem % tiles_y;
    rem /= tiles_y;
    const int xt = rem % tiles_x;
    const long b = rem / tiles_x;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int W = 2 * cz + 1;
    // first fine point of the tile (halo included)
    const int fx = 2 * xt * CX + a.off[0] - 1, fy = 2 * yt * CY + a.off[1] - 1,
              fz = 2 * zt * cz + a.off[2] - 1;
    const __amdgpu_buffer_rsrc_t src =
        brsrc(a.in + b * a.in_grid, (unsigned)(a.in_grid * sizeof(TI)));
    // wrapped index along an axis (-1: zero) and its Bloch factor, applied
    // after those of the axes before
    auto wrap = [&](int i, int c, double2& f, bool& ph) {
        if (i >= 0 && i < a.ni[c]) return i;
        if (!a.periodic[c]) return -1;
        while (i < 0) {
            i += a.ni[c];
            f = ph ? cmul(a.ph[c][1], f) : a.ph[c][1];
            ph = true;
        }
        while (i >= a.ni[c]) {
            i -= a.ni[c];
            f = ph ? cmul(a.ph[c][0], f) : a.ph[c][0];
            ph = true;
        }
        return i;
    };
    // byte offset of a fine row, BXM_OOB if it is zero
    auto row_at = [&](int r, double2& f, bool& ph) -> unsigned {
        f = make_double2(1.0, 0.0);
        ph = false;
        const int x = wrap(fx + r / RY, 0, f, ph);
        const int y = wrap(fy + r % RY, 1, f, ph);
        return x < 0 || y < 0
                   ? BXM_OOB
                   : ((unsigned)x * a.ni[1] + (unsigned)y) * a.ni[2] *
                         (unsigned)sizeof(TI);
    };
    // the z factor comes last: f_z (f_y f_x)
    auto put = [&](int r, int z, TI v, double2 f, bool ph, double2 g,
                   bool gph) {
        if constexpr (CPLX)
            if (ph || gph)
                v = apply_phase(v, ph ? (gph ? cmul(g, f) : f) : g);
        E[r * RT_P + z] = narrow<T, TI>(v);
    };
    double2 zf = make_double2(1.0, 0.0);
    bool zph = false;
    const int zw = lane < W ? wrap(fz + lane, 2, zf, zph) : -1;
    const unsigned zo = zw < 0 ? BXM_OOB : (unsigned)zw * sizeof(TI);
    // two rounds of loads per wave
    constexpr int J = (ROWS + 3) / 4, JU = (J + 1) / 2;
    for (int j0 = 0; j0 < J; j0 += JU) {
        TI v[JU];
        double2 rf[JU];
        bool rph[JU];
        cfor<JU>([&](auto j) {
            const int r = min(w + 4 * (j0 + j), ROWS - 1);
            const unsigned ro = row_at(r, rf[j], rph[j]);
            v[j] = bload<TI>(src, ro == BXM_OOB || zo == BXM_OOB
                                      ? BXM_OOB : ro + zo);
        });
        cfor<JU>([&](auto j) {
            const int r = min(w + 4 * (j0 + j), ROWS - 1);
            if (lane < W) put(r, lane, v[j], rf[j], rph[j], zf, zph);
        });
    }
    if (W > 64 && t < ROWS) {  // the last point of each full row
        double2 f, g = make_double2(1.0, 0.0);
        bool ph, gph = false;
        const int z = wrap(fz + 64, 2, g, gph);
        const unsigned ro = row_at(t, f, ph);
        put(t, 64,
            bload<TI>(src, ro == BXM_OOB || z < 0
                               ? BXM_OOB : ro + (unsigned)z * sizeof(TI)),
            f, ph, g, gph);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CX * CY * RT_CZ / 256; k++) {
        const int id = t + 256 * k;
        const int z = id % RT_CZ, y = id / RT_CZ % CY, x = id / (RT_CZ * CY);
        const int oz = zt * cz + z, oy = yt * CY + y, ox = xt * CX + x;
        if (z >= cz || oz >= a.no[2] || oy >= a.no[1] || ox >= a.no[0])
            continue;
        const T* p = E + (2 * x * RY + 2 * y) * RT_P + 2 * z;
        T px[3];
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
            T py[3];
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const T* q = p + (dx * RY + dy) * RT_P;
                const T zp = q[2] + q[0];
                py[dy] = (S)0.5 * fmac(q[1], (S)0.5, zp);
            }
            px[dx] = (S)0.5 * fmac(py[1], (S)0.5, py[2] + py[0]);
        }
        const T v = (S)0.5 * fmac(px[1], (S)0.5, px[2] + px[0]);
        f3store<T, EPI, TI>(
            a, b * a.out_grid + ((long)ox * a.no[1] + oy) * a.no[2] + oz, v);
    }
}

template <typename T, int EPI, typename TI>
__global__ void __launch_bounds__(256) k_interp2(F3Args<T, TI> a)
{
    typedef typename ScalarOf<T>::type S;
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= a.total) return;
    long b;
    int o0, o1, o2;
    flat_split(gid, a.total, a.out_grid, a.no[1], a.no[2], b, o0, o1, o2);
    const int q0 = o0 + a.skip0[0], q1 = o1 + a.skip0[1], q2 = o2 + a.skip0[2];
    const int c0 = (q0 >> 1) + a.off[0], c1 = (q1 >> 1) + a.off[1],
              c2 = (q2 >> 1) + a.off[2];
    const int n0 = (q0 & 1) + 1, n1 = (q1 & 1) + 1, n2 = (q2 & 1) + 1;
    const TI* __restrict__ g = a.in + b * a.in_grid;
    T vx[2];
#pragma unroll
    for (int dx = 0; dx < 2; dx++) {
        if (dx >= n0) break;
        T vy[2];
#pragma unroll
        for (int dy = 0; dy < 2; dy++) {
            if (dy >= n1) break;
            T vz = f3load(a, g, c0 + dx, c1 + dy, c2);
            if (n2 == 2)
                vz = (S)0.5 * (vz + f3load(a, g, c0 + dx, c1 + dy, c2 + 1));
            vy[dy] = vz;
        }
        vx[dx] = (n1 == 2) ? (S)0.5 * (vy[0] + vy[1]) : vy[0];
    }
    const T v = (n0 == 2) ? (S)0.5 * (vx[0] + vx[1]) : vx[0];
    f3store<T, EPI, TI>(a, gid, v);
}

// value of interpolated output point (o0, o1, o2) of grid g
template <typename T, typename TI>
__device__ inline T interp2_point(const F3Args<T, TI>& a,
                                  const TI* __restrict__ g, int o0, int o1,
                                  int o2)
{
    typedef typename ScalarOf<T>::type S;
    const int q0 = o0 + a.skip0[0], q1 = o1 + a.skip0[1], q2 = o2 + a.skip0[2];
    const int c0 = (q0 >> 1) + a.off[0], c1 = (q1 >> 1) + a.off[1],
              c2 = (q2 >> 1) + a.off[2];
    const int n0 = (q0 & 1) + 1, n1 = (q1 & 1) + 1, n2 = (q2 & 1) + 1;
    T vx[2];
#pragma unroll
    for (int dx = 0; dx < 2; dx++) {
        if (dx >= n0) break;
        T vy[2];
#pragma unroll
        for (int dy = 0; dy < 2; dy++) {
            if (dy >= n1) break;
            T vz = f3load(a, g, c0 + dx, c1 + dy, c2);
            if (n2 == 2)
                vz = (S)0.5 * (vz + f3load(a, g, c0 + dx, c1 + dy, c2 + 1));
            vy[dy] = vz;
        }
        vx[dx] = (n1 == 2) ? (S)0.5 * (vy[0] + vy[1]) : vy[0];
    }
    return (n0 == 2) ? (S)0.5 * (vx[0] + vx[1]) : vx[0];
}

// Two neighbouring outputs along z per thread (even output rows): the
// index arithmetic is shared and the coarse values both need are loaded
// once
template <typename T, int EPI, typename TI>
__global__ void __launch_bounds__(256) k_interp2p(F3Args<T, TI> a)
{
    const long gp = (long)blockIdx.x * 256 + threadIdx.x;
    if (2 * gp >= a.total) return;
    const long gid = 2 * gp;
    long b;
    int o0, o1, o2;
    flat_split(gid, a.total, a.out_grid, a.no[1], a.no[2], b, o0, o1, o2);
    const TI* __restrict__ g = a.in + b * a.in_grid;
    const T v0 = interp2_point(a, g, o0, o1, o2);
    const T v1 = interp2_point(a, g, o0, o1, o2 + 1);
    f3store<T, EPI, TI>(a, gid, v0);
    f3store<T, EPI, TI>(a, gid + 1, v1);
}

template <typename T, typename TI>
static F3Args<T, TI> f3args(const XferPlan& p, const BC& bc, const void* in,
                            void* out, long nin, const XEpiArgs& ea)
{
    F3Args<T, TI> a;
    a.in = (const TI*)in;
    a.out = (T*)out;
    a.out2 = (T*)ea.out2;
    a.base = (const T*)ea.base;
    for (int c = 0; c < 3; c++) {
        a.ni[c] = p.nin[c];
        a.no[c] = p.nout[c];
        a.off[c] = p.ax[c].off;
        a.skip0[c] = p.ax[c].skip0;
        a.periodic[c] = bc.periodic[c];
        a.ph[c][0] = bc.phase[c][0];
        a.ph[c][1] = bc.phase[c][1];
    }
    a.in_grid = (long)p.nin[0] * p.nin[1] * p.nin[2];
    a.out_grid = (long)p.nout[0] * p.nout[1] * p.nout[2];
    a.total = a.out_grid * nin;
    a.negate = ea.negate;
    a.alpha = ea.alpha;
    return a;
}

template <typename T, int EPI, typename TI>
static int launch_rtile_t(const XferPlan& p, const BC& bc, const void* in,
                          void* out, long nin, const XEpiArgs& ea,
                          hipStream_t s)
{
    const F3Args<T, TI> a = f3args<T, TI>(p, bc, in, out, nin, ea);
    if (p.interpolate || p.K != 2 ||
        a.in_grid * (long)sizeof(TI) >= (1L << 31)) {
        set_error("tiled restriction: not for this transfer");
        return ENOTSUP_;
    }
    const int tz = ceil_div(a.no[2], RT_CZ), cz = ceil_div(a.no[2], tz);
    const int ty = ceil_div(a.no[1], RtTile<T>::CY);
    const int tx = ceil_div(a.no[0], RtTile<T>::CX);
    const long nb = (long)tz * ty * tx * nin;
    if (nb <= 0) return OK;
    if (nb > 0x7fffffffL) {
        set_error("transfer: too many blocks");
        return ENOTSUP_;
    }
    hipLaunchKernelGGL((k_restrict_tile<T, EPI, TI>), dim3((unsigned)nb),
                       dim3(256), 0, s, a, cz, tz, ty, tx, (int)nb);
    GFD_LAUNCH_CHECK();
    return OK;
}

template <typename T, typename TI = T>
static int launch_rtile(const XferPlan& p, const BC& bc, const void* in,
                        void* out, long nin, const XEpiArgs& ea,
                        hipStream_t s)
{
    switch (ea.epi) {
    case XEPI_PLAIN: return launch_rtile_t<T, XEPI_PLAIN, TI>(p, bc, in, out, nin, ea, s);
    case XEPI_NEG: return launch_rtile_t<T, XEPI_NEG, TI>(p, bc, in, out, nin, ea, s);
    case XEPI_SCALE2: return launch_rtile_t<T, XEPI_SCALE2, TI>(p, bc, in, out, nin, ea, s);
    case XEPI_SUBFROM: return launch_rtile_t<T, XEPI_SUBFROM, TI>(p, bc, in, out, nin, ea, s);
    }
    set_error("transfer: bad epilogue %d", ea.epi);
    return EINVAL_;
}

static int launch_restrict_tile(const XferPlan& p, int dtype, const BC& bc,
                                const void* in, void* out, long nin,
                                const XEpiArgs& ea, hipStream_t s)
{
    switch (dtype) {
    case 0: return launch_rtile<double>(p, bc, in, out, nin, ea, s);
    case 1: return launch_rtile<double2>(p, bc, in, out, nin, ea, s);
    case 2: return ea.in_wide ? launch_rtile<float, double>(p, bc, in, out, nin, ea, s)
                              : launch_rtile<float>(p, bc, in, out, nin, ea, s);
    case 3: return ea.in_wide ? launch_rtile<float2, double2>(p, bc, in, out, nin, ea, s)
                              : launch_rtile<float2>(p, bc, in, out, nin, ea, s);
    }
    set_error("transfer: bad dtype %d", dtype);
    return EINVAL_;
}

template <typename T, int EPI, typename TI>
static int launch_fused2_t(const XferPlan& p, const BC& bc, const void* in,
                           void* out, long nin, const XEpiArgs& ea,
                           hipStream_t s)
{
    const F3Args<T, TI> a = f3args<T, TI>(p, bc, in, out, nin, ea);
    const long nb = (a.total + 255) / 256;
    if (nb <= 0) return OK;
    if (nb > 0x7fffffffL) {
        set_error("transfer: too many blocks");
        return ENOTSUP_;
    }
    if (p.interpolate && p.nout[2] % 2 == 0)
        hipLaunchKernelGGL((k_interp2p<T, EPI, TI>),
                           dim3((unsigned)((a.total / 2 + 255) / 256)),
                           dim3(256), 0, s, a);
    else if (p.interpolate)
        hipLaunchKernelGGL((k_interp2<T, EPI, TI>), dim3((unsigned)nb),
                           dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_restrict2<T, EPI, TI>), dim3((unsigned)nb),
                           dim3(256), 0, s, a);
    GFD_LAUNCH_CHECK();
    return OK;
}

template <typename T, typename TI = T>
static int launch_fused2(const XferPlan& p, const BC& bc, const void* in,
                         void* out, long nin, const XEpiArgs& ea,
                         hipStream_t s)
{
    switch (ea.epi) {
    case XEPI_PLAIN: return launch_fused2_t<T, XEPI_PLAIN, TI>(p, bc, in, out, nin, ea, s);
    case XEPI_NEG: return launch_fused2_t<T, XEPI_NEG, TI>(p, bc, in, out, nin, ea, s);
    case XEPI_SCALE2: return launch_fused2_t<T, XEPI_SCALE2, TI>(p, bc, in, out, nin, ea, s);
    case XEPI_SUBFROM: return launch_fused2_t<T, XEPI_SUBFROM, TI>(p, bc, in, out, nin, ea, s);
    }
    set_error("transfer: bad epilogue %d", ea.epi);
    return EINVAL_;
}

long xfer_scratch_elems(const XferPlan& p, long nin, bool three)
{
    // output of the y pass, and of a z pass of its own
    return (long)p.nin[0] * (p.nout[1] + (three ? p.nin[1] : 0)) *
           p.nout[2] * nin;
}

// z and y passes of a separable transfer in one launch: a block stages the
// input rows under cy x zt outputs of one x plane in LDS, z-transforms them
// there and writes the y transforms of the result.  As two launches the z
// pass read each point K + 1 times through L1 and its result, as large as
// half the input, went through memory.  The 1-D sums are those of the x pass.
// Bound by the chain of a block (load, z, y; LDS reads of 7 values a point).
// Two passes before -> this and x, K = 6: restriction of 4 real grids of 96^3
// 25.4 -> 22.1 us, 32 of them 150 -> 122, one of 48^3 16.6 -> 8.4; staged
// columns in order instead of even / odd: 24.2.  Interpolation of 4 complex
// grids of 96^3 at K = 8 50.7 -> 38.6 (marching 112).  Threads take columns
// side by side: with a wave per row 35 grids of 200x60x24 took 64 us at K = 4
// (now 41, two passes 42).  Where a tile's halo is large against it, at K = 8
// above all, two passes stay the faster ones (56 boxes of 30x40x150 53 us, 69
// here), so both are timed per shape.
template <typename T>
struct ZyArgs {
    const T* in;
    T* out;
    int n0, ni1, ni2, no1, no2;  // planes; rows and columns in and out
    int cy, zt;                  // outputs of a block
    int ry, rz;                  // staged rows and columns at most
    int tiles_y, tiles_z, nblocks;
    int off[2], skip0[2], periodic[2];  // y, z
    double2 ph[2][2];
};

template <int K, bool INTERP>
__device__ __host__ inline int zy_first(int i, int off, int skip0)
{
    return INTERP ? ((i + skip0) >> 1) + off - (K / 2 - 1)
                  : 2 * i + off - (K - 1);
}

template <int K, bool INTERP>
__device__ __host__ inline int zy_last(int i, int off, int skip0)
{
    return INTERP ? ((i + skip0) >> 1) + off + K / 2
                  : 2 * i + off + (K - 1);
}

// output from the input at its centre p, neighbours s apart
template <typename T, int K, bool INTERP>
__device__ inline T zy_point(const T* p, int s, bool odd)
{
    typedef typename ScalarOf<T>::type S;
    if constexpr (!INTERP) {
        T acc = p[0];
#pragma unroll
        for (int m = 0; m < K / 2; m++) {
            const int j = (2 * m + 1) * s;
            acc = fmac(acc, (S)W<K>::w[m], p[j] + p[-j]);
        }
        return (S)0.5 * acc;
    } else {
        if (!odd) return p[0];
        T acc = (S)W<K>::w[0] * (p[0] + p[s]);
#pragma unroll
        for (int m = 1; m < K / 2; m++)
            acc = fmac(acc, (S)W<K>::w[m], p[-m * s] + p[(1 + m) * s]);
        return acc;
    }
}

template <typename T, int K, bool INTERP>
__global__ void __launch_bounds__(256) k_xfer_zy(ZyArgs<T> a)
{
    typedef typename ScalarOf<T>::type S;
    extern __shared__ __align__(16) char zy_lds[];
    T* const E = reinterpret_cast<T*>(zy_lds);  // staged rows
    T* const Z = E + a.ry * a.rz;               // their z transforms
    int rem = xcd_remap(blockIdx.x, a.nblocks);
    const int zt = rem % a.tiles_z;
    rem /= a.tiles_z;
    const int yt = rem % a.tiles_y;
    const long pl = rem / a.tiles_y;
    const int t = threadIdx.x;
    const int oy0 = yt * a.cy, oy1 = min(oy0 + a.cy, a.no1);
    const int oz0 = zt * a.zt, oz1 = min(oz0 + a.zt, a.no2);
    const int iy0 = zy_first<K, INTERP>(oy0, a.off[0], a.skip0[0]);
    const int iz0 = zy_first<K, INTERP>(oz0, a.off[1], a.skip0[1]);
    const int ny = zy_last<K, INTERP>(oy1 - 1, a.off[0], a.skip0[0]) - iy0 + 1;
    const int nz = zy_last<K, INTERP>(oz1 - 1, a.off[1], a.skip0[1]) - iz0 + 1;
    const T* __restrict__ g = a.in + pl * a.ni1 * a.ni2;
    // staged column: for a restriction the even ones, then the odd ones, so
    // that lanes next to each other read next to each other
    const int half = (a.rz + 1) / 2;
    auto col = [&](int z) {
        return INTERP ? z : (z & 1) * half + (z >> 1);
    };
    // index inside the array (-1: zero) and its Bloch factor
    auto wrap = [&](int i, int n, int c, double2& f, bool& ph) {
        f = make_double2(1.0, 0.0);
        ph = false;
        if (i >= 0 && i < n) return i;
        if (!a.periodic[c]) return -1;
        while (i < 0) {
            i += n;
            f = ph ? cmul(a.ph[c][1], f) : a.ph[c][1];
            ph = true;
        }
        while (i >= n) {
            i -= n;
            f = ph ? cmul(a.ph[c][0], f) : a.ph[c][0];
            ph = true;
        }
        return i;
    };
    // A thread keeps one column of the staged rows, as many rows side by side
    // as the block holds.
    constexpr int JU = sizeof(T) == 16 ? 8 : 12;  // loads in flight
    {
        const int side = 256 / nz;
        const int r0 = t / nz, z = t - r0 * nz;
        double2 f, fy;
        bool ph, py;
        const int iz = wrap(iz0 + z, a.ni2, 1, f, ph);
        for (int j0 = r0 < side ? r0 : ny; j0 < ny; j0 += side * JU) {
            T v[JU];
#pragma unroll
            for (int j = 0; j < JU; j++) {
                v[j] = zero_of<T>();
                const int r = j0 + side * j;
                if (r >= ny) continue;
                const int iy = wrap(iy0 + r, a.ni1, 0, fy, py);
                if (iy >= 0 && iz >= 0) v[j] = g[(long)iy * a.ni2 + iz];
            }
#pragma unroll
            for (int j = 0; j < JU; j++) {
                const int r = j0 + side * j;
                if constexpr (XIsCplx<T>::value)
                    if (iz >= 0 && ph) v[j] = cmul(f, v[j]);
                if (r < ny) E[r * a.rz + col(z)] = v[j];
            }
        }
    }
    __syncthreads();
    constexpr int BACK = INTERP ? K / 2 - 1 : K - 1;  // centre in its window
    const int noz = oz1 - oz0;
    const int dr = 256 / noz, dz = 256 % noz;
    for (int r = t / noz, z = t % noz; r < ny;) {
        T v;
        if constexpr (INTERP) {
            const int c = zy_first<K, INTERP>(oz0 + z, a.off[1],
                                              a.skip0[1]) - iz0 + BACK;
            v = zy_point<T, K, INTERP>(E + r * a.rz + c, 1,
                                       (oz0 + z + a.skip0[1]) & 1);
        } else {
            // centre: staged column 2z + K - 1, neighbours: even columns
            const T* p = E + r * a.rz + z + K / 2 - 1;
            T acc = p[half];
#pragma unroll
            for (int m = 0; m < K / 2; m++)
                acc = fmac(acc, (S)W<K>::w[m], p[m + 1] + p[-m]);
            v = (S)0.5 * acc;
        }
        if constexpr (XIsCplx<T>::value) {
            double2 f;
            bool ph;
            wrap(iy0 + r, a.ni1, 0, f, ph);
            if (ph) v = cmul(f, v);
        }
        Z[r * a.zt + z] = v;
        r += dr;
        z += dz;
        if (z >= noz) {
            z -= noz;
            r++;
        }
    }
    __syncthreads();
    T* __restrict__ o = a.out + pl * a.no1 * a.no2;
    const int side = 256 / noz;
    const int z = t % noz;
    for (int oy = oy0 + (t < side * noz ? t / noz : a.cy); oy < oy1;
         oy += side) {
        const int c =
            zy_first<K, INTERP>(oy, a.off[0], a.skip0[0]) - iy0 + BACK;
        o[(long)oy * a.no2 + oz0 + z] = zy_point<T, K, INTERP>(
            Z + c * a.zt + z, a.zt, (oy + a.skip0[0]) & 1);
    }
}

// Outputs of a block: rows in equal parts of at most 64 columns (48 in
// complex FP64, 128 when interpolating) by as many rows as leave 1024 blocks
// and fit 64 KB of LDS; four rows always do (53 KB in complex FP64 at K = 8).
template <typename T, int K, bool INTERP>
static int launch_zy(const XferPlan& p, const BC& bc, const T* in, T* out,
                     long nin, hipStream_t s)
{
    ZyArgs<T> a;
    a.in = in;
    a.out = out;
    a.n0 = p.nin[0];
    a.ni1 = p.nin[1];
    a.ni2 = p.nin[2];
    a.no1 = p.nout[1];
    a.no2 = p.nout[2];
    for (int c = 0; c < 2; c++) {
        a.off[c] = p.ax[c + 1].off;
        a.skip0[c] = p.ax[c + 1].skip0;
        a.periodic[c] = bc.periodic[c + 1];
        a.ph[c][0] = bc.phase[c + 1][0];
        a.ph[c][1] = bc.phase[c + 1][1];
    }
    const long planes = (long)a.n0 * nin;
    if (planes <= 0 || a.no1 <= 0 || a.no2 <= 0) return OK;
    a.tiles_z = ceil_div(a.no2, INTERP ? 128 : sizeof(T) == 16 ? 48 : 64);
    a.zt = ceil_div(a.no2, a.tiles_z);
    // inputs under c outputs
    auto span = [](int c) {
        return INTERP ? c / 2 + K : 2 * (c - 1) + 2 * (K - 1) + 1;
    };
    a.rz = span(a.zt);
    size_t lds = 0;
    for (a.cy = INTERP ? 32 : 16;; a.cy /= 2) {
        a.tiles_y = ceil_div(a.no1, a.cy);
        a.ry = span(a.cy);
        lds = (size_t)a.ry * (a.rz + a.zt) * sizeof(T);
        if (a.cy == 4 || (lds <= 65536 &&
                          planes * a.tiles_y * a.tiles_z >= 1024))
            break;
    }
    const long nb = planes * a.tiles_y * a.tiles_z;
    if (nb > 0x7fffffffL) {
        set_error("transfer: too many blocks");
        return ENOTSUP_;
    }
    a.nblocks = (int)nb;
    hipLaunchKernelGGL((k_xfer_zy<T, K, INTERP>), dim3((unsigned)nb),
                       dim3(256), lds, s, a);
    GFD_LAUNCH_CHECK();
    return OK;
}

template <typename T, int AX, int K, bool INTERP, int EPI>
static int launch_pass(XArgs<T> a, hipStream_t s)
{
    const long nb = (a.total + 255) / 256;
    if (nb <= 0) return OK;
    if (nb > 0x7fffffffL) {
        set_error("transfer: too many blocks");
        return ENOTSUP_;
    }
    hipLaunchKernelGGL((k_xfer1d<T, AX, K, INTERP, EPI>), dim3((unsigned)nb),
                       dim3(256), 0, s, a);
    GFD_LAUNCH_CHECK();
    return OK;
}

template <typename T, int K, bool INTERP>
static int launch_pass_epi(XArgs<T> a, int epi, hipStream_t s)
{
    switch (epi) {
    case XEPI_PLAIN: return launch_pass<T, 0, K, INTERP, XEPI_PLAIN>(a, s);
    case XEPI_NEG: return launch_pass<T, 0, K, INTERP, XEPI_NEG>(a, s);
    case XEPI_SCALE2: return launch_pass<T, 0, K, INTERP, XEPI_SCALE2>(a, s);
    case XEPI_SUBFROM: return launch_pass<T, 0, K, INTERP, XEPI_SUBFROM>(a, s);
    }
    set_error("transfer: bad epilogue %d", epi);
    return EINVAL_;
}

// three: z and y in a launch each, z's result behind y's in the work space;
// else both in one (k_xfer_zy).
template <typename T, int K, bool INTERP>
static int run_transfer(const XferPlan& p, const BC& bc, const void* in,
                        void* out, long nin, void* scratch, bool three,
                        const XEpiArgs& ea, hipStream_t s)
{
    auto pass = [&](int ax, const T* from, T* to) {
        XArgs<T> a;
        a.in = from;
        a.out = to;
        a.out2 = (T*)ea.out2;
        a.base = (const T*)ea.base;
        // the axes after this one are done, those before it are not
        for (int c = 0; c < 3; c++) a.d[c] = c < ax ? p.nin[c] : p.nout[c];
        a.ilen = p.nin[ax];
        a.istride = ax == 2   ? 1
                    : ax == 1 ? (long)p.nout[2]
                              : (long)p.nout[1] * p.nout[2];
        a.out_grid = (long)a.d[0] * a.d[1] * a.d[2];
        a.in_grid = a.out_grid / a.d[ax] * a.ilen;
        a.total = a.out_grid * nin;
        a.off = p.ax[ax].off;
        a.skip0 = p.ax[ax].skip0;
        a.periodic = bc.periodic[ax];
        a.ph_hi = bc.phase[ax][0];
        a.ph_lo = bc.phase[ax][1];
        a.negate = ea.negate;
        a.alpha = ea.alpha;
        return a;
    };
    T* const zy = (T*)scratch;
    T* const z = zy + (long)p.nin[0] * p.nout[1] * p.nout[2] * nin;
    if (three) {
        GFD_TRY((launch_pass<T, 2, K, INTERP, XEPI_PLAIN>(
            pass(2, (const T*)in, z), s)));
        GFD_TRY((launch_pass<T, 1, K, INTERP, XEPI_PLAIN>(pass(1, z, zy), s)));
    } else {
        GFD_TRY((launch_zy<T, K, INTERP>(p, bc, (const T*)in, zy, nin, s)));
    }
    return launch_pass_epi<T, K, INTERP>(pass(0, zy, (T*)out), ea.epi, s);
}

template <typename T>
static int run_transfer_k(const XferPlan& p, const BC& bc, const void* in,
                          void* out, long nin, void* scratch, bool three,
                          const XEpiArgs& ea, hipStream_t s)
{
    const bool I = p.interpolate != 0;
    switch (p.K) {
    case 2: return I ? run_transfer<T, 2, true>(p, bc, in, out, nin, scratch, three, ea, s)
                     : run_transfer<T, 2, false>(p, bc, in, out, nin, scratch, three, ea, s);
    case 4: return I ? run_transfer<T, 4, true>(p, bc, in, out, nin, scratch, three, ea, s)
                     : run_transfer<T, 4, false>(p, bc, in, out, nin, scratch, three, ea, s);
    case 6: return I ? run_transfer<T, 6, true>(p, bc, in, out, nin, scratch, three, ea, s)
                     : run_transfer<T, 6, false>(p, bc, in, out, nin, scratch, three, ea, s);
    case 8: return I ? run_transfer<T, 8, true>(p, bc, in, out, nin, scratch, three, ea, s)
                     : run_transfer<T, 8, false>(p, bc, in, out, nin, scratch, three, ea, s);
    }
    set_error("transfer: unsupported K=%d", p.K);
    return EINVAL_;
}

static bool g_xfer_force_passes = false;
static bool g_xfer_three = false;  // forced passes in a launch each
static bool g_xfer_march = true;

bool xfer_passes_forced() { return g_xfer_force_passes; }

void xfer_force_passes(bool on, bool three)
{
    g_xfer_force_passes = on;
    g_xfer_three = on && three;
}
void xfer_set_march(bool on) { g_xfer_march = on; }

// ------------------------------------------------- kernel choice (timed)
//
// Per transfer shape (plan, data type, batch, input width) the faster of
// the x-marching kernel and the one-point / separable-pass kernels, timed
// once on the call's own input into a scratch output.  Without an entry the
// marching kernel runs.

struct XKey {
    int v[12];
    bool operator<(const XKey& o) const
    {
        return std::lexicographical_compare(v, v + 12, o.v, o.v + 12);
    }
};

static std::mutex g_xc_mu;
// 0 marching, 1 other kernels, 2 tiled K = 2 restriction, 3 (K > 2) z and y
// passes in a launch each
static std::map<XKey, int> g_xchoice;
static std::atomic<bool> g_xfer_tile{false};  // tiled wherever it fits

void xfer_set_tile(bool on) { g_xfer_tile = on; }

static bool g_xtune = true;

void xfer_set_autotune(bool on)
{
    std::lock_guard<std::mutex> lk(g_xc_mu);
    g_xtune = on;
    if (!on) g_xchoice.clear();
}

static XKey xkey(const XferPlan& p, int dtype, long nin, int in_wide)
{
    XKey k;
    k.v[0] = p.K;
    k.v[1] = p.interpolate;
    for (int c = 0; c < 3; c++) {
        k.v[2 + c] = p.nin[c];
        k.v[5 + c] = p.nout[c];
    }
    k.v[8] = dtype;
    k.v[9] = (int)std::min<long>(nin, 0x7fffffffL);
    k.v[10] = in_wide;
    k.v[11] = 0;
    return k;
}

static int launch_other(const XferPlan& p, int dtype, const BC& bc,
                        const void* in, void* out, long nin, void* scratch,
                        bool three, const XEpiArgs& ea, hipStream_t stream);

bool xfer_needs_tuning(const XferPlan& p, int dtype, long nin, int in_wide)
{
    std::lock_guard<std::mutex> lk(g_xc_mu);
    return g_xtune && g_xfer_march && !g_xfer_force_passes &&
           g_xchoice.find(xkey(p, dtype, nin, in_wide)) == g_xchoice.end();
}

bool xfer_wants_three(const XferPlan& p, int dtype, long nin, int in_wide)
{
    if (g_xfer_three) return true;
    if (p.K == 2) return false;
    std::lock_guard<std::mutex> lk(g_xc_mu);
    auto it = g_xchoice.find(xkey(p, dtype, nin, in_wide));
    return it == g_xchoice.end() ? g_xtune : it->second == 3;
}

int xfer_tune(const XferPlan& p, int dtype, const BC& bc, const void* in,
              void* tune_out, long nin, void* scratch, bool room,
              int in_wide, hipStream_t s)
{
    XEpiArgs ea;
    ea.in_wide = in_wide;
    hipEvent_t e0, e1;
    GFD_CHECK_HIP(hipEventCreate(&e0));
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        set_error("transfer tuner: hipEventCreate failed");
        return EHIP;
    }
    float best = 1e30f;
    int choice = 0;
    for (int c = 0; c < 4; c++) {
        if (c == 2 && (p.K != 2 || p.interpolate)) continue;
        if (c == 3 && (p.K == 2 || !room)) continue;
        auto run = [&]() {
            return c == 0 ? launch_transfer_march(p, dtype, bc, in, tune_out,
                                                  nin, ea, s)
                 : c == 2 ? launch_restrict_tile(p, dtype, bc, in, tune_out,
                                                 nin, ea, s)
                          : launch_other(p, dtype, bc, in, tune_out, nin,
                                         scratch, c == 3, ea, s);
        };
        if (run() != OK) {  // this kernel cannot take the shape
            set_error("");
            continue;
        }
        (void)hipEventRecord(e0, s);
        int st = OK;
        for (int r = 0; r < 3 && st == OK; r++) st = run();
        (void)hipEventRecord(e1, s);
        if (hipEventSynchronize(e1) != hipSuccess || st != OK) {
            (void)hipGetLastError();
            set_error("");
            continue;
        }
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        if (ms < best) {
            best = ms;
            choice = c;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    std::lock_guard<std::mutex> lk(g_xc_mu);
    g_xchoice[xkey(p, dtype, nin, in_wide)] = choice;
    return OK;
}

int launch_transfer(const XferPlan& p, int dtype, const BC& bc,
                    const void* in, void* out, long nin, void* scratch,
                    bool room, const XEpiArgs& ea, hipStream_t stream)
{
    if (ea.in_wide && (p.K != 2 || (dtype != 2 && dtype != 3))) {
        set_error("transfer: FP64 input only for FP32 data and K = 2");
        return EINVAL_;
    }
    bool march = g_xfer_march && !g_xfer_force_passes;
    bool tile = g_xfer_tile && p.K == 2 && !p.interpolate;
    bool three = g_xfer_three;
    if (march && !tile) {
        std::lock_guard<std::mutex> lk(g_xc_mu);
        auto it = g_xchoice.find(xkey(p, dtype, nin, ea.in_wide));
        if (it != g_xchoice.end()) {
            march = it->second == 0;
            tile = it->second == 2;
            three = it->second == 3;
        }
    }
    if (tile) {
        const int st =
            launch_restrict_tile(p, dtype, bc, in, out, nin, ea, stream);
        if (st != ENOTSUP_) return st;
        set_error("");
    }
    if (march) {
        // the x-marching fused kernel (xfer_march.hip), any K
        const int st =
            launch_transfer_march(p, dtype, bc, in, out, nin, ea, stream);
        if (st != ENOTSUP_) return st;
        set_error("");
    }
    return launch_other(p, dtype, bc, in, out, nin, scratch, three && room,
                        ea, stream);
}

// the one-point-per-thread K = 2 kernels, or the separable passes
static int launch_other(const XferPlan& p, int dtype, const BC& bc,
                        const void* in, void* out, long nin, void* scratch,
                        bool three, const XEpiArgs& ea, hipStream_t stream)
{
    if (dtype == 3 && p.K != 2) {
        set_error("transfer: complex64 data only for K = 2");
        return ENOTSUP_;
    }
    // K = 2 on the separable passes only when forced and given their work
    // space (caller-owned work spaces are sized for the fused kernel)
    if (p.K == 2 &&
        (!g_xfer_force_passes || dtype == 3 || ea.in_wide || !scratch)) {
        if (dtype == 0)
            return launch_fused2<double>(p, bc, in, out, nin, ea, stream);
        if (dtype == 1)
            return launch_fused2<double2>(p, bc, in, out, nin, ea, stream);
        if (dtype == 2)
            return ea.in_wide
                       ? launch_fused2<float, double>(p, bc, in, out, nin, ea,
                                                      stream)
                       : launch_fused2<float>(p, bc, in, out, nin, ea, stream);
        if (dtype == 3)
            return ea.in_wide
                       ? launch_fused2<float2, double2>(p, bc, in, out, nin,
                                                        ea, stream)
                       : launch_fused2<float2>(p, bc, in, out, nin, ea,
                                               stream);
    }
    if (dtype == 0)
        return run_transfer_k<double>(p, bc, in, out, nin, scratch, three, ea,
                                      stream);
    if (dtype == 1)
        return run_transfer_k<double2>(p, bc, in, out, nin, scratch, three, ea,
                                      stream);
    if (dtype == 2)
        return run_transfer_k<float>(p, bc, in, out, nin, scratch, three, ea,
                                      stream);
    set_error("transfer: bad dtype %d", dtype);
    return EINVAL_;
}

}  // namespace gfd
