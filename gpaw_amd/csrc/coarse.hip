// LDS-resident coarse V-cycle (see coarse.h).
//
// The coarse levels of a multigrid hierarchy hold few points (24^3 FP32 =
// 54 KB) but cost a dozen launches each when run like the fine levels;
// here one workgroup of 1024 threads keeps every coarse level's arrays in
// LDS and runs the down-sweep (Jacobi pre-smoothing, residual, restriction),
// the coarsest-level sweeps and the up-sweep (interpolation + correction,
// post-smoothing) with barriers between passes.  The arithmetic per point
// is that of the global kernels: Jacobi (1 - w) e + w (r - sum_nb) / c0,
// residual (c0 e + sum_nb) - r, and the K = 2 transfer weights in the
// same association order (z innermost, then y, then x).
#include "../../include/gpaw_fd.h"
#include "coarse.h"

#include <algorithm>
#include <atomic>
#include <cmath>

#include "stencil_dev.h"

namespace gfd {

// index along an axis with periodic wrap, -1 outside a zero boundary
__device__ inline int cw(int i, int n, int periodic)
{
    if (i >= 0 && i < n) return i;
    if (!periodic) return -1;
    i %= n;
    if (i < 0) i += n;
    return i;
}

template <typename T>
__device__ inline T cat(const T* a, int idx)
{
    return idx >= 0 ? a[idx] : zero_of<T>();
}

// Threads own columns (i1, i2) of a level and march along x; when a plane
// has fewer columns than threads, the x range is split between `parts`
// thread groups.
struct CWork {
    int q0, qstep;   // first column, column stride
    int x0, x1;      // x range
};

__device__ inline CWork cwork(int plane, int n0)
{
    CWork w;
    const int nt = blockDim.x, t = threadIdx.x;
    const int parts = plane >= nt ? 1 : min(nt / plane, n0);
    if (t >= parts * (plane >= nt ? nt : plane)) {
        w.q0 = plane;  // idle
        w.qstep = 1;
        w.x0 = w.x1 = 0;
        return w;
    }
    if (plane >= nt) {
        w.q0 = t;
        w.qstep = nt;
        w.x0 = 0;
        w.x1 = n0;
    } else {
        const int part = t / plane;
        w.q0 = t % plane;
        w.qstep = plane;  // one column
        w.x0 = part * n0 / parts;
        w.x1 = (part + 1) * n0 / parts;
    }
    return w;
}

// plane offsets of the z and y neighbours of column q (-1: zero boundary)
struct CCol {
    int zo[2][CMAXR];
    int yo[2][CMAXR];
};

__device__ inline void ccol(const CLevel& L, int q, CCol& c)
{
    const int n2 = L.n[2];
    const int i2 = q % n2, i1 = q / n2;
#pragma unroll
    for (int k = 1; k <= CMAXR; k++) {
#pragma unroll
        for (int sg = 0; sg < 2; sg++) {
            const int d = sg ? -k : k;
            const int j = cw(i2 + d, n2, L.periodic[2]);
            c.zo[sg][k - 1] = j < 0 ? -1 : i1 * n2 + j;
            const int y = cw(i1 + d, L.n[1], L.periodic[1]);
            c.yo[sg][k - 1] = y < 0 ? -1 : y * n2 + i2;
        }
    }
}

// off-centre stencil terms at (i0, column q): z, then y, then x
template <typename T>
__device__ inline T cneigh(const T* e, const CLevel& L, const CCol& c,
                           int q, int i0, int plane)
{
    typedef typename ScalarOf<T>::type S;
    const T* row = e + i0 * plane;
    T acc = zero_of<T>();
    if (L.has[2]) {
#pragma unroll
        for (int k = 1; k <= CMAXR; k++) {
            if (k > L.R) break;
            acc = fmac(acc, (S)L.cp[2][k - 1], cat(row, c.zo[0][k - 1]));
            acc = fmac(acc, (S)L.cm[2][k - 1], cat(row, c.zo[1][k - 1]));
        }
    }
    if (L.has[1]) {
#pragma unroll
        for (int k = 1; k <= CMAXR; k++) {
            if (k > L.R) break;
            acc = fmac(acc, (S)L.cp[1][k - 1], cat(row, c.yo[0][k - 1]));
            acc = fmac(acc, (S)L.cm[1][k - 1], cat(row, c.yo[1][k - 1]));
        }
    }
    if (L.has[0]) {
#pragma unroll
        for (int k = 1; k <= CMAXR; k++) {
            if (k > L.R) break;
            const int xp = cw(i0 + k, L.n[0], L.periodic[0]);
            const int xm = cw(i0 - k, L.n[0], L.periodic[0]);
            acc = fmac(acc, (S)L.cp[0][k - 1],
                       cat(e, xp < 0 ? -1 : xp * plane + q));
            acc = fmac(acc, (S)L.cm[0][k - 1],
                       cat(e, xm < 0 ? -1 : xm * plane + q));
        }
    }
    return acc;
}

// `sweeps` Jacobi sweeps on level L; bit `lbit` of cur says which of A / B
// holds the current iterate.
template <typename T>
__device__ void crelax(T* sm, const CLevel& L, const T* rl, int sweeps,
                       unsigned& cur, int lbit)
{
    typedef typename ScalarOf<T>::type S;
    const int plane = L.n[1] * L.n[2];
    const CWork w = cwork(plane, L.n[0]);
    for (int s = 0; s < sweeps; s++) {
        const bool inb = (cur >> lbit) & 1u;
        const T* src = sm + (inb ? L.b : L.a);
        T* dst = sm + (inb ? L.a : L.b);
        for (int q = w.q0; q < plane; q += w.qstep) {
            CCol c;
            ccol(L, q, c);
            for (int i0 = w.x0; i0 < w.x1; i0++) {
                const int p = i0 * plane + q;
                const T acc = cneigh(src, L, c, q, i0, plane);
                dst[p] = ((S)1.0 - (S)L.w) * src[p] +
                         (S)L.w * (rl[p] - acc) / (S)L.c0;
            }
            if (w.qstep == plane) break;
        }
        __syncthreads();
        cur ^= 1u << lbit;
    }
}

// `steps` steps of Chebyshev iteration for A e = r with the Jacobi
// preconditioner D = c0 (Saad, Iterative Methods for Sparse Linear
// Systems, 2nd ed., Alg. 12.1): with the eigenvalues of D^-1 A in
// [lo, hi], theta = (hi + lo) / 2, delta = (hi - lo) / 2, sigma =
// theta / delta, z = D^-1 (r - A e):
//   d_0 = z_0 / theta,  rho_0 = 1 / sigma
//   rho_k = 1 / (2 sigma - rho_{k-1}),
//   d_k = rho_k rho_{k-1} d_{k-1} + (2 rho_k / delta) z_k,  e += d_k.
// After m steps the error is p_m(D^-1 A) e_0 with p_m the scaled
// Chebyshev polynomial, |p_m| <= 2 ((sqrt k - 1) / (sqrt k + 1))^m on
// [lo, hi] (k = hi / lo), where m Jacobi sweeps give (1 - w lo)^m.
template <typename T>
__device__ void ccheb(T* sm, const CLevel& L, const T* rl, int steps,
                      unsigned& cur, int lbit)
{
    typedef typename ScalarOf<T>::type S;
    const int plane = L.n[1] * L.n[2];
    const CWork w = cwork(plane, L.n[0]);
    T* D = sm + L.dbuf;
    const double theta = 0.5 * (L.lam_hi + L.lam_lo);
    const double delta = 0.5 * (L.lam_hi - L.lam_lo);
    const double sigma = theta / delta;
    double rho = 1.0 / sigma;
    for (int s = 0; s < steps; s++) {
        double ca = 0.0, cb = 1.0 / theta;
        if (s > 0) {
            const double rn = 1.0 / (2.0 * sigma - rho);
            ca = rn * rho;
            cb = 2.0 * rn / delta;
            rho = rn;
        }
        const S a = (S)ca, bq = (S)cb;
        const bool inb = (cur >> lbit) & 1u;
        const T* src = sm + (inb ? L.b : L.a);
        T* dst = sm + (inb ? L.a : L.b);
        for (int q = w.q0; q < plane; q += w.qstep) {
            CCol c;
            ccol(L, q, c);
            for (int i0 = w.x0; i0 < w.x1; i0++) {
                const int p = i0 * plane + q;
                const T acc = cneigh(src, L, c, q, i0, plane);
                const T z = (rl[p] - acc) / (S)L.c0 - src[p];
                const T dd = s > 0 ? fmac(bq * z, a, D[p]) : bq * z;
                D[p] = dd;
                dst[p] = src[p] + dd;
            }
            if (w.qstep == plane) break;
        }
        __syncthreads();
        cur ^= 1u << lbit;
    }
}

template <typename T>
__global__ void __launch_bounds__(1024)
k_coarse(const CGrid* __restrict__ grids, const T* __restrict__ rhs,
         T* __restrict__ out)
{
    typedef typename ScalarOf<T>::type S;
    extern __shared__ __align__(16) unsigned char csm_raw[];
    T* sm = reinterpret_cast<T*>(csm_raw);
    // the descriptor in LDS: its fields are re-read after every barrier,
    // which from global memory costs a round trip each time
    __shared__ CGrid G;
    {
        const int* src = reinterpret_cast<const int*>(grids + blockIdx.x);
        int* dst = reinterpret_cast<int*>(&G);
        for (int i = threadIdx.x; i < (int)(sizeof(CGrid) / sizeof(int));
             i += blockDim.x)
            dst[i] = src[i];
        __syncthreads();
    }
    const int nl = G.nlev;
    const T* r0 = rhs + G.rhs_off;
    unsigned cur = 0;   // bit l: level l's iterate is in B

    // first level of the block: e = 0, and its rhs staged in LDS when the
    // plan left room (every pass then stays in LDS)
    {
        const CLevel& L = G.lev[0];
        const int n = L.n[0] * L.n[1] * L.n[2];
        for (int p = threadIdx.x; p < n; p += blockDim.x) {
            sm[L.a + p] = zero_of<T>();
            if (L.r >= 0) sm[L.r + p] = r0[p];
        }
        __syncthreads();
    }
    // down
    for (int l = 0; l + 1 < nl; l++) {
        const CLevel& L = G.lev[l];
        const CLevel& N = G.lev[l + 1];
        const T* rl = L.r >= 0 ? sm + L.r : r0;
        crelax(sm, L, rl, L.pre, cur, l);
        const bool inb = (cur >> l) & 1u;
        const T* E = sm + (inb ? L.b : L.a);
        T* W = sm + (inb ? L.a : L.b);
        const int plane = L.n[1] * L.n[2];
        {
            const CWork w = cwork(plane, L.n[0]);
            for (int q = w.q0; q < plane; q += w.qstep) {
                CCol c;
                ccol(L, q, c);
                for (int i0 = w.x0; i0 < w.x1; i0++) {
                    const int p = i0 * plane + q;
                    const T acc = cneigh(E, L, c, q, i0, plane);
                    W[p] = fmac(acc, (S)L.c0, E[p]) - rl[p];
                }
                if (w.qstep == plane) break;
            }
        }
        __syncthreads();
        // restriction of W into N's rhs; N's iterate starts at zero
        const int nplane = N.n[1] * N.n[2];
        const CWork w = cwork(nplane, N.n[0]);
        for (int q = w.q0; q < nplane; q += w.qstep) {
            const int o2 = q % N.n[2], o1 = q / N.n[2];
            int off[3][3];  // [dy + 1][dz + 1]: plane offset in L, -1: zero
#pragma unroll
            for (int dy = -1; dy <= 1; dy++) {
                const int y = cw(2 * o1 + L.roff[1] + dy, L.n[1],
                                 L.periodic[1]);
#pragma unroll
                for (int dz = -1; dz <= 1; dz++) {
                    const int z = cw(2 * o2 + L.roff[2] + dz, L.n[2],
                                     L.periodic[2]);
                    off[dy + 1][dz + 1] =
                        (y < 0 || z < 0) ? -1 : y * L.n[2] + z;
                }
            }
            for (int o0 = w.x0; o0 < w.x1; o0++) {
                T px[3];
#pragma unroll
                for (int dx = -1; dx <= 1; dx++) {
                    const int x = cw(2 * o0 + L.roff[0] + dx, L.n[0],
                                     L.periodic[0]);
                    T py[3];
#pragma unroll
                    for (int dy = 0; dy < 3; dy++) {
                        T a0 = zero_of<T>(), am = a0, ap = a0;
                        if (x >= 0) {
                            const T* row = W + x * plane;
                            am = cat(row, off[dy][0]);
                            a0 = cat(row, off[dy][1]);
                            ap = cat(row, off[dy][2]);
                        }
                        py[dy] = (S)0.5 * fmac(a0, (S)0.5, ap + am);
                    }
                    px[dx + 1] = (S)0.5 * fmac(py[1], (S)0.5, py[2] + py[0]);
                }
                const int qq = o0 * nplane + q;
                sm[N.r + qq] = (S)0.5 * fmac(px[1], (S)0.5, px[2] + px[0]);
                sm[N.a + qq] = zero_of<T>();
            }
            if (w.qstep == nplane) break;
        }
        __syncthreads();
    }
    // coarsest
    {
        const CLevel& L = G.lev[nl - 1];
        const T* rl = L.r >= 0 ? sm + L.r : r0;
        if (L.cheb)
            ccheb(sm, L, rl, L.post, cur, nl - 1);
        else
            crelax(sm, L, rl, L.post, cur, nl - 1);
    }
    // up
    for (int l = nl - 2; l >= 0; l--) {
        const CLevel& L = G.lev[l];
        const CLevel& N = G.lev[l + 1];
        const T* EN = sm + (((cur >> (l + 1)) & 1u) ? N.b : N.a);
        T* E = sm + (((cur >> l) & 1u) ? L.b : L.a);
        const int plane = L.n[1] * L.n[2];
        const int nplane = N.n[1] * N.n[2];
        const CWork w = cwork(plane, L.n[0]);
        for (int q = w.q0; q < plane; q += w.qstep) {
            const int o2 = q % L.n[2], o1 = q / L.n[2];
            const int q1 = o1 + L.iskip0[1], q2 = o2 + L.iskip0[2];
            const int c1 = (q1 >> 1) + L.ioff[1], c2 = (q2 >> 1) + L.ioff[2];
            const int m1 = (q1 & 1) + 1, m2 = (q2 & 1) + 1;
            int off[2][2];  // [dy][dz]: plane offset in N, -1: zero
#pragma unroll
            for (int dy = 0; dy < 2; dy++) {
                const int y = cw(c1 + dy, N.n[1], N.periodic[1]);
#pragma unroll
                for (int dz = 0; dz < 2; dz++) {
                    const int z = cw(c2 + dz, N.n[2], N.periodic[2]);
                    off[dy][dz] = (y < 0 || z < 0) ? -1 : y * N.n[2] + z;
                }
            }
            for (int o0 = w.x0; o0 < w.x1; o0++) {
                const int q0 = o0 + L.iskip0[0];
                const int c0 = (q0 >> 1) + L.ioff[0];
                const int m0 = (q0 & 1) + 1;
                T vx[2];
#pragma unroll
                for (int dx = 0; dx < 2; dx++) {
                    if (dx >= m0) break;
                    const int x = cw(c0 + dx, N.n[0], N.periodic[0]);
                    T vy[2];
#pragma unroll
                    for (int dy = 0; dy < 2; dy++) {
                        if (dy >= m1) break;
                        T vz = zero_of<T>(), vz1 = vz;
                        if (x >= 0) {
                            const T* row = EN + x * nplane;
                            vz = cat(row, off[dy][0]);
                            if (m2 == 2) vz1 = cat(row, off[dy][1]);
                        }
                        if (m2 == 2) vz = (S)0.5 * (vz + vz1);
                        vy[dy] = vz;
                    }
                    vx[dx] = (m1 == 2) ? (S)0.5 * (vy[0] + vy[1]) : vy[0];
                }
                const T v = (m0 == 2) ? (S)0.5 * (vx[0] + vx[1]) : vx[0];
                const int p = o0 * plane + q;
                E[p] = E[p] - v;
            }
            if (w.qstep == plane) break;
        }
        __syncthreads();
        const T* rl = L.r >= 0 ? sm + L.r : r0;
        crelax(sm, L, rl, L.post, cur, l);
    }
    // result
    {
        const CLevel& L = G.lev[0];
        const T* E = sm + ((cur & 1u) ? L.b : L.a);
        const int n = L.n[0] * L.n[1] * L.n[2];
        T* o = out + G.out_off;
        for (int p = threadIdx.x; p < n; p += blockDim.x) o[p] = E[p];
    }
}

// ------------------------------------------------- nearest-neighbour form
//
// k_coarse1: the same solve for levels with 7-point (radius 1) stencils,
// every coarse level of the standard hierarchies.  A thread owns one x
// segment of one (y, z) column: its iterate and right-hand side stay in
// registers over all sweeps of a stage, the four in-plane neighbour offsets
// (and zeroed coefficients in place of a zero boundary's branches) are
// formed once per stage, and only the four in-plane neighbours and the
// segment's two end neighbours are read from LDS.  The stages of a level
// are fused with the transfers that feed them: restriction into the
// registers of the first sweep (from zero: the scaled right-hand side),
// interpolation into the start of the post-sweeps.  A level of at most 64
// segments runs in one wave without barriers.
//
// What bounds it: the serial chain of barriers and LDS round trips, not
// bytes.  k_coarse forms every neighbour index (with divisions by the row
// length, and one by c0 per point) in every sweep.  Measured: FP64 12^3 ..
// 3^3 of a 48^3 cycle 85 -> 26 us; the batched FP32 levels of twelve grids
// (up to 10 x 20 x 20) 94 -> 30 us; FP32 24^3 .. 3^3 74 us against some 190
// us as launches with k_coarse from 12^3 down.
// Threads of a block, and the longest segment (FP32 first levels up to 24
// planes; in FP64 the 128 registers of a 1024-thread block leave 76 bytes of
// scratch per thread at 12 already, which the 26 us above include).  Segments beyond C1_X only on the first
// level (a deeper one has at most a quarter of its columns) and not with
// the Chebyshev iteration.
constexpr int C1_NT = 1024, C1_X = 12, C1_XFIRST = 24;

template <typename T>
struct CSeg {
    int p0, len;             // first point, points (0: idle thread)
    int plane;
    int dzp, dzm, dyp, dym;  // neighbour offsets (0 with a zero coefficient)
    int xlo, xhi;            // points before / after the segment
    T czp, czm, cyp, cym, cxp, cxm, cxlo, cxhi;
    T c0, w1, wc;
    int x0, i1, i2;
};

template <typename T>
__device__ inline CSeg<T> cseg(const CLevel& L)
{
    CSeg<T> s;
    const int n0 = L.n[0], n1 = L.n[1], n2 = L.n[2];
    s.plane = n1 * n2;
    const int t = threadIdx.x;
    const int part = t / s.plane, q = t - part * s.plane;
    s.i1 = q / n2;
    s.i2 = q - s.i1 * n2;
    s.x0 = 0;
    s.len = 0;
    s.p0 = 0;
    if (part < L.parts) {
        s.x0 = part * n0 / L.parts;
        s.len = (part + 1) * n0 / L.parts - s.x0;
        s.p0 = s.x0 * s.plane + q;
    }
    auto off = [&](int i, int d, int n, int periodic, int stride, T c,
                   int& o) -> T {
        const int j = cw(i + d, n, periodic);
        o = j < 0 ? 0 : (j - i) * stride;
        return j < 0 ? (T)0 : c;
    };
    const T z = (T)0;
    s.czp = off(s.i2, 1, n2, L.periodic[2], 1, L.has[2] ? (T)L.cp[2][0] : z, s.dzp);
    s.czm = off(s.i2, -1, n2, L.periodic[2], 1, L.has[2] ? (T)L.cm[2][0] : z, s.dzm);
    s.cyp = off(s.i1, 1, n1, L.periodic[1], n2, L.has[1] ? (T)L.cp[1][0] : z, s.dyp);
    s.cym = off(s.i1, -1, n1, L.periodic[1], n2, L.has[1] ? (T)L.cm[1][0] : z, s.dym);
    s.cxp = L.has[0] ? (T)L.cp[0][0] : z;
    s.cxm = L.has[0] ? (T)L.cm[0][0] : z;
    s.xlo = s.xhi = 0;
    s.cxlo = s.cxhi = z;
    if (s.len > 0) {
        int o;
        s.cxlo = off(s.x0, -1, n0, L.periodic[0], s.plane, s.cxm, o);
        s.xlo = s.p0 + o;
        const int xl = s.x0 + s.len - 1, pl = s.p0 + (s.len - 1) * s.plane;
        s.cxhi = off(xl, 1, n0, L.periodic[0], s.plane, s.cxp, o);
        s.xhi = pl + o;
    }
    s.c0 = (T)L.c0;
    s.w1 = (T)(1.0 - L.w);
    s.wc = (T)(L.w / L.c0);
    return s;
}

// f(i, acc): acc = off-centre stencil terms of the segment's point i (z,
// then y, then x), the iterate's own values in e, the rest from src.  f may
// overwrite e[i].
template <typename T, int XL, typename F>
__device__ __forceinline__ void cseg_pass(const CSeg<T>& s, const T* src, T* e, F&& f)
{
    T below = src[s.xlo];
    const T above = src[s.xhi];
    // the running point is opaque: its neighbour addresses would otherwise
    // be hoisted out of the sweeps, five registers for every point
    int p = s.p0;
    if (XL > 2) asm volatile("" : "+v"(p));
    cfor<XL>([&](auto ic) {
        constexpr int i = ic;
        if (i < s.len) {
            const T* row = src + p;
            T acc = (T)0;
            acc = fmac(acc, s.czp, row[s.dzp]);
            acc = fmac(acc, s.czm, row[s.dzm]);
            acc = fmac(acc, s.cyp, row[s.dyp]);
            acc = fmac(acc, s.cym, row[s.dym]);
            const bool last = i + 1 == s.len;
            const T up = last || i + 1 == XL ? above : e[(i + 1) % XL];
            acc = fmac(acc, last ? s.cxhi : s.cxp, up);
            acc = fmac(acc, i == 0 ? s.cxlo : s.cxm, below);
            below = e[i];
            f(ic, acc);
        }
        p += s.plane;
        // bounds the loads the scheduler moves ahead (registers)
        if (XL > 4 && (i & (sizeof(T) == 8 ? 1 : 3)) == 0)
            __builtin_amdgcn_sched_barrier(0);
    });
}

template <bool ONE>
__device__ inline void csync()
{
    if (ONE) {
        // one wave: LDS operations of a wave complete in order, only the
        // compiler has to keep theirs
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

template <typename T, int XL>
__device__ inline void cseg_write(const CSeg<T>& s, T* dst, const T* e)
{
    int p = s.p0;
    if (XL > 2) asm volatile("" : "+v"(p));
    cfor<XL>([&](auto i) {
        if (i < s.len) dst[p] = e[i];
        p += s.plane;
    });
}

// `n` Jacobi sweeps on e (already in the LDS buffer `cur` and synchronised);
// the last one is left in registers only with `keep`
template <typename T, int XL, bool ONE>
__device__ __forceinline__ void cseg_sweeps(const CSeg<T>& s, const CLevel& L, T* sm,
                                   const T* r, T* e, int n, int& cur,
                                   bool keep)
{
    for (int k = 0; k < n; k++) {
        cseg_pass<T, XL>(s, sm + (cur ? L.b : L.a), e, [&](auto i, T acc) {
            e[i] = fmac(s.w1 * e[i], s.wc, r[i] - acc);
        });
        if (keep && k + 1 == n) return;
        cur ^= 1;
        cseg_write<T, XL>(s, sm + (cur ? L.b : L.a), e);
        csync<ONE>();
    }
}

template <typename T, int XL, bool ONE>
__device__ __forceinline__ void cdown(T* sm, const CGrid& G, int l, unsigned curs,
                      const T* r0, T* out)
{
    typedef typename ScalarOf<T>::type S;
    const CLevel& L = G.lev[l];
    const CSeg<T> s = cseg<T>(L);
    const bool coarsest = l + 1 == G.nlev;
    T r[XL], e[XL];
    if (XL > C1_X || l == 0) {
        cfor<XL>([&](auto i) {
            r[i] = i < s.len ? r0[s.p0 + i * s.plane] : (T)0;
        });
    } else {
        // restriction of the finer level's residual
        const CLevel& F = G.lev[l - 1];
        const T* W = sm + (((curs >> (l - 1)) & 1u) ? F.a : F.b);
        const int fplane = F.n[1] * F.n[2];
        int off[3][3];  // [dy + 1][dz + 1]: plane offset in F, -1: zero
#pragma unroll
        for (int dy = -1; dy <= 1; dy++) {
            const int y = cw(2 * s.i1 + F.roff[1] + dy, F.n[1], F.periodic[1]);
#pragma unroll
            for (int dz = -1; dz <= 1; dz++) {
                const int z =
                    cw(2 * s.i2 + F.roff[2] + dz, F.n[2], F.periodic[2]);
                off[dy + 1][dz + 1] = (y < 0 || z < 0) ? -1 : y * F.n[2] + z;
            }
        }
        auto fplane_sum = [&](int x) -> T {
            x = cw(x, F.n[0], F.periodic[0]);
            if (x < 0) return (T)0;
            const T* row = W + x * fplane;
            T py[3];
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
                py[dy] = (S)0.5 * fmac(cat(row, off[dy][1]), (S)0.5,
                                       cat(row, off[dy][2]) +
                                           cat(row, off[dy][0]));
            return (S)0.5 * fmac(py[1], (S)0.5, py[2] + py[0]);
        };
        const int xf = 2 * s.x0 + F.roff[0];
        T lo = s.len > 0 ? fplane_sum(xf - 1) : (T)0;
        if (XL > 2) __builtin_amdgcn_sched_barrier(0);
        cfor<XL>([&](auto i) {
            r[i] = (T)0;
            if (i < s.len) {
                const T mid = fplane_sum(xf + 2 * i);
                const T hi = fplane_sum(xf + 2 * i + 1);
                r[i] = (S)0.5 * fmac(mid, (S)0.5, hi + lo);
                lo = hi;
            }
            if (XL > 2) __builtin_amdgcn_sched_barrier(0);
        });
        if (!coarsest) cseg_write<T, XL>(s, sm + L.r, r);
    }
    int cur = 0;
    const int n = coarsest ? L.post : L.pre;
    if (XL <= C1_X && coarsest && L.cheb) {
        // update array: in registers for short segments, else in LDS
        constexpr bool DREG = XL <= 3;
        T d[DREG ? XL : 1];
        T* dl = sm + L.dbuf + s.p0;
        const S ic = (S)(1.0 / L.c0);
        const S b0 = (S)G.cheb_b[0];
        cfor<XL>([&](auto i) {
            e[i] = n > 0 ? b0 * (r[i] * ic) : (T)0;
            if constexpr (DREG) d[i] = e[i];
            else if (i < s.len) dl[i * s.plane] = e[i];
        });
        cseg_write<T, XL>(s, sm + L.a, e);
        csync<ONE>();
        for (int k = 1; k < n; k++) {
            const S ca = (S)G.cheb_a[k], cb = (S)G.cheb_b[k];
            cseg_pass<T, XL>(s, sm + (cur ? L.b : L.a), e, [&](auto i, T acc) {
                const T z = (r[i] - acc) * ic - e[i];
                if constexpr (DREG) {
                    d[i] = fmac(cb * z, ca, d[i]);
                    e[i] = e[i] + d[i];
                } else {
                    const T dd = fmac(cb * z, ca, dl[i * s.plane]);
                    dl[i * s.plane] = dd;
                    e[i] = e[i] + dd;
                }
            });
            cur ^= 1;
            cseg_write<T, XL>(s, sm + (cur ? L.b : L.a), e);
            csync<ONE>();
        }
    } else {
        // the first sweep from e = 0 is the scaled right-hand side
        cfor<XL>([&](auto i) { e[i] = n > 0 ? s.wc * r[i] : (T)0; });
        cseg_write<T, XL>(s, sm + L.a, e);
        csync<ONE>();
        cseg_sweeps<T, XL, ONE>(s, L, sm, r, e, n - 1, cur, false);
    }
    if (coarsest) {
        if (l == 0) cseg_write<T, XL>(s, out, e);
    } else {
        // residual over e; the iterate stays in its LDS array
        cseg_pass<T, XL>(s, sm + (cur ? L.b : L.a), e, [&](auto i, T acc) {
            e[i] = fmac(acc, s.c0, e[i]) - r[i];
        });
        cseg_write<T, XL>(s, sm + (cur ? L.a : L.b), e);
        csync<ONE>();
    }
}

template <typename T, int XL, bool ONE>
__device__ __forceinline__ void cup(T* sm, const CGrid& G, int l, unsigned curs,
                    const T* r0, T* out)
{
    typedef typename ScalarOf<T>::type S;
    const CLevel& L = G.lev[l];
    const CLevel& N = G.lev[l + 1];
    const CSeg<T> s = cseg<T>(L);
    int cur = (curs >> l) & 1u;
    T r[XL], e[XL];
    const T* rl = l == 0 ? r0 : sm + L.r;
    const T* es = sm + (cur ? L.b : L.a);
    cfor<XL>([&](auto i) {
        r[i] = e[i] = (T)0;
        if (i < s.len) {
            r[i] = rl[s.p0 + i * s.plane];
            e[i] = es[s.p0 + i * s.plane];
        }
    });
    {
        const T* EN = sm + (((curs >> (l + 1)) & 1u) ? N.b : N.a);
        const int nplane = N.n[1] * N.n[2];
        const int q1 = s.i1 + L.iskip0[1], q2 = s.i2 + L.iskip0[2];
        const int c1 = (q1 >> 1) + L.ioff[1], c2 = (q2 >> 1) + L.ioff[2];
        const bool h1 = q1 & 1, h2 = q2 & 1;
        int off[2][2];  // [dy][dz]: plane offset in N, -1: zero
#pragma unroll
        for (int dy = 0; dy < 2; dy++) {
            const int y = cw(c1 + dy, N.n[1], N.periodic[1]);
#pragma unroll
            for (int dz = 0; dz < 2; dz++) {
                const int z = cw(c2 + dz, N.n[2], N.periodic[2]);
                off[dy][dz] = (y < 0 || z < 0) ? -1 : y * N.n[2] + z;
            }
        }
        auto nplane_val = [&](int x) -> T {
            x = cw(x, N.n[0], N.periodic[0]);
            if (x < 0) return (T)0;
            const T* row = EN + x * nplane;
            T v0 = cat(row, off[0][0]);
            if (h2) v0 = (S)0.5 * (v0 + cat(row, off[0][1]));
            if (h1) {
                T v1 = cat(row, off[1][0]);
                if (h2) v1 = (S)0.5 * (v1 + cat(row, off[1][1]));
                v0 = (S)0.5 * (v0 + v1);
            }
            return v0;
        };
        cfor<XL>([&](auto i) {
            if (i < s.len) {
                const int q0 = s.x0 + i + L.iskip0[0];
                const int c0 = (q0 >> 1) + L.ioff[0];
                T v = nplane_val(c0);
                if (q0 & 1) v = (S)0.5 * (v + nplane_val(c0 + 1));
                e[i] = e[i] - v;
            }
            if (XL > 2) __builtin_amdgcn_sched_barrier(0);
        });
    }
    const int n = L.post;
    if (n > 0) {
        cseg_write<T, XL>(s, sm + (cur ? L.b : L.a), e);
        csync<ONE>();
        cseg_sweeps<T, XL, ONE>(s, L, sm, r, e, n, cur, l == 0);
    } else if (l > 0) {
        cseg_write<T, XL>(s, sm + (cur ? L.b : L.a), e);
        csync<ONE>();
    }
    if (l == 0) cseg_write<T, XL>(s, out, e);
}

// One stage of level l with the segment length as a constant; afterwards
// every thread notes which array holds the level's iterate (one swap per
// sweep that writes LDS: the first sweep from zero does not swap).
template <typename T, int XM, bool UP>
__device__ __forceinline__ void cstage(T* sm, const CGrid& G, int l, unsigned& curs,
                              const T* r0, T* out)
{
    const CLevel& L = G.lev[l];
#define GFD_CS(XX, ONE)                                                     \
    do {                                                                    \
        if (UP) cup<T, XX, ONE>(sm, G, l, curs, r0, out);                   \
        else cdown<T, XX, ONE>(sm, G, l, curs, r0, out);                    \
    } while (0)
    const int xl = L.xl;
    if (L.onewave) {
        if (threadIdx.x < 64) {
            if (xl <= 1) GFD_CS(1, true);
            else GFD_CS(3, true);
        }
        __syncthreads();
    } else if (xl <= 1) GFD_CS(1, false);
    else if (xl <= 2) GFD_CS(2, false);
    else if (xl <= 3) GFD_CS(3, false);
    else if (xl <= 4) GFD_CS(4, false);
    else if (xl <= 6) GFD_CS(6, false);
    else if (xl <= 12) GFD_CS(12, false);
    else {
        if constexpr (XM > 12) GFD_CS(XM, false);
    }
#undef GFD_CS
    const int swaps = UP ? L.post
                         : (l + 1 == G.nlev ? L.post : L.pre) - 1;
    if (swaps > 0 && (swaps & 1)) curs ^= 1u << l;
}

template <typename T, int XM>
__global__ void __launch_bounds__(C1_NT)
k_coarse1(const CGrid* __restrict__ grids, const T* __restrict__ rhs,
          T* __restrict__ out)
{
    extern __shared__ __align__(16) unsigned char csm_raw[];
    T* sm = reinterpret_cast<T*>(csm_raw);
    __shared__ CGrid G;
    {
        const int* src = reinterpret_cast<const int*>(grids + blockIdx.x);
        int* dst = reinterpret_cast<int*>(&G);
        for (int i = threadIdx.x; i < (int)(sizeof(CGrid) / sizeof(int));
             i += C1_NT)
            dst[i] = src[i];
        __syncthreads();
    }
    const T* r0 = rhs + G.rhs_off;
    T* o = out + G.out_off;
    const int nl = G.nlev;
    unsigned curs = 0;  // bit l: level l's iterate is in its array b
    for (int l = 0; l < nl; l++) cstage<T, XM, false>(sm, G, l, curs, r0, o);
    for (int l = nl - 2; l >= 0; l--)
        cstage<T, XM, true>(sm, G, l, curs, r0, o);
}

static bool g_cheb = true;

void coarse_set_cheb(bool on) { g_cheb = on; }
bool coarse_cheb_enabled() { return g_cheb; }

bool cheb_bounds(const CLevel& L, double* lo, double* hi)
{
    if (L.R != 1 || L.c0 == 0.0) return false;
    // lambda(theta) = 1 + sum_c g_c(theta_c), g_c = (cp e^{i theta} +
    // cm e^{-i theta}) / c0 = 2 cp cos(theta) / c0 for cp = cm
    double gmin[3], gnext[3], gmax[3];
    for (int c = 0; c < 3; c++) {
        const double cp = L.has[c] ? L.cp[c][0] : 0.0;
        const double cm = L.has[c] ? L.cm[c][0] : 0.0;
        if (cp != cm) return false;
        const int n = L.n[c];
        gmin[c] = 1e300;
        gnext[c] = 1e300;
        gmax[c] = -1e300;
        for (int j = 0; j < n; j++) {
            const double th = L.periodic[c] ? 2.0 * M_PI * j / n
                                            : M_PI * (j + 1) / (n + 1);
            const double g = 2.0 * cp * std::cos(th) / L.c0;
            gmax[c] = std::max(gmax[c], g);
            if (g < gmin[c]) {
                gnext[c] = gmin[c];
                gmin[c] = g;
            } else if (g < gnext[c]) {
                gnext[c] = g;
            }
        }
    }
    double smin = 1.0, smax = 1.0;
    for (int c = 0; c < 3; c++) {
        smin += gmin[c];
        smax += gmax[c];
    }
    double l0 = smin;
    if (l0 <= 1e-9 * smax) {
        // the constant mode of a periodic operator (eigenvalue 0): the
        // smallest nonzero one moves one axis to its next mode
        l0 = 1e300;
        for (int c = 0; c < 3; c++)
            if (gnext[c] < 1e299) l0 = std::min(l0, smin + gnext[c] - gmin[c]);
    }
    if (!(l0 > 0.0) || !(smax > l0) || l0 >= 1e299) return false;
    // rounding and non-exact modes: a lower bound too low only slows the
    // iteration, an upper bound too low lets the top modes grow
    *lo = 0.9 * l0;
    *hi = 1.05 * smax;
    return true;
}

static bool plan1_level(CLevel& L, int xmax)
{
    const int plane = L.n[1] * L.n[2], n0 = L.n[0];
    if (L.R != 1 || plane > C1_NT) return false;
    auto split = [&](int threads) {
        L.parts = std::min(threads / plane, n0);
        L.xl = (n0 + L.parts - 1) / L.parts;
        L.parts = (n0 + L.xl - 1) / L.xl;
    };
    L.onewave = 0;
    if (plane <= 64) {
        split(64);
        L.onewave = L.xl <= 3;
    }
    if (!L.onewave) split(C1_NT);
    return L.xl <= (L.cheb ? C1_X : xmax);
}

bool coarse_plan1(CGrid* grids, int G, int dtype)
{
    for (int g = 0; g < G; g++) {
        CGrid& c = grids[g];
        const CLevel& C = c.lev[c.nlev - 1];
        if (!C.cheb) continue;
        if (C.post > CCHEB) return false;
        // ccheb's recurrence, tabulated
        const double theta = 0.5 * (C.lam_hi + C.lam_lo);
        const double delta = 0.5 * (C.lam_hi - C.lam_lo);
        const double sigma = theta / delta;
        double rho = 1.0 / sigma;
        c.cheb_a[0] = 0.0;
        c.cheb_b[0] = 1.0 / theta;
        for (int k = 1; k < C.post; k++) {
            const double rn = 1.0 / (2.0 * sigma - rho);
            c.cheb_a[k] = rn * rho;
            c.cheb_b[k] = 2.0 * rn / delta;
            rho = rn;
        }
    }
    for (int g = 0; g < G; g++)
        for (int i = 0; i < grids[g].nlev; i++)
            if (!plan1_level(grids[g].lev[i],
                             i == 0 && dtype == 2 ? C1_XFIRST : C1_X))
                return false;
    return true;
}

int launch_coarse(const CGrid* d_grids, int G, size_t lds_bytes, int dtype,
                  const void* rhs, void* out, bool one, hipStream_t s)
{
    if (G <= 0) return OK;
    if (lds_bytes > COARSE_LDS_MAX) {
        set_error("coarse solve: %zu bytes of LDS requested", lds_bytes);
        return EINVAL_;
    }
    typedef void (*KF)(const CGrid*, const float*, float*);
    typedef void (*KD)(const CGrid*, const double*, double*);
    const KF kf = one ? k_coarse1<float, C1_XFIRST> : k_coarse<float>;
    const KD kd = one ? k_coarse1<double, C1_X> : k_coarse<double>;
    const void* fn = dtype == 2 ? (const void*)kf : (const void*)kd;
    // above the default 64 KB of LDS: opted into once per kernel
    static std::atomic<bool> raised[2][2];
    std::atomic<bool>& up = raised[dtype == 2][one];
    if (lds_bytes > 64 * 1024 && !up) {
        const hipError_t e = hipFuncSetAttribute(
            fn, hipFuncAttributeMaxDynamicSharedMemorySize,
            (int)COARSE_LDS_MAX);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            set_error("coarse solve: LDS attribute failed (%s)",
                      hipGetErrorString(e));
            return ENOTSUP_;
        }
        up = true;
    }
    if (dtype == 2)
        hipLaunchKernelGGL(kf, dim3(G), dim3(1024), lds_bytes, s, d_grids,
                           (const float*)rhs, (float*)out);
    else
        hipLaunchKernelGGL(kd, dim3(G), dim3(1024), lds_bytes, s, d_grids,
                           (const double*)rhs, (double*)out);
    GFD_LAUNCH_CHECK();
    return OK;
}

}  // namespace gfd

extern "C" int gfd_coarse_cheb_bounds(const int* n, const int* periodic,
                                      const double* cp, double c0,
                                      double* lo, double* hi)
{
    if (!n || !periodic || !cp || !lo || !hi) {
        gfd::set_error("gfd_coarse_cheb_bounds: null argument");
        return gfd::EINVAL_;
    }
    gfd::CLevel L{};
    L.R = 1;
    L.c0 = c0;
    for (int c = 0; c < 3; c++) {
        if (n[c] < 1) {
            gfd::set_error("gfd_coarse_cheb_bounds: bad shape");
            return gfd::EINVAL_;
        }
        L.n[c] = n[c];
        L.periodic[c] = periodic[c];
        L.has[c] = cp[c] != 0.0;
        L.cp[c][0] = L.cm[c][0] = cp[c];
    }
    if (!gfd::cheb_bounds(L, lo, hi)) {
        gfd::set_error("gfd_coarse_cheb_bounds: no bounds for this stencil");
        return gfd::ENOTSUP_;
    }
    return gfd::OK;
}
