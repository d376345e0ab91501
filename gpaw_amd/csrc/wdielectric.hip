// The dielectric operator eps lap + grad eps . grad (weighted stencils: one
// symmetric axis stencil over all three axes, then one antisymmetric stencil
// per axis, real or Bloch-complex data), applied or swept by weighted
// Jacobi (c/bmgs/wfd.cpp, c/bmgs/wrelax.cpp).
//
// k_wdiel marches along x like k_dirmarch (dirmarch_kernel.h), staging every
// plane of a tile with its halo once in LDS, but with a ring of R + 2 planes:
// all four sums of an output point are formed in one step, when the plane R
// ahead of it has arrived (x terms from a register queue of 2R + 1 centre
// values), because each is multiplied by its own weight of that point.  The
// block order runs over the grids of the batch first: their blocks of one
// tile read its four weights from the same XCD's L2.
//
// What bounds it: latency and traffic together (32 bytes of weights beside 16
// of data per point; by counters 279 MiB fetched for 135, 4.5 TB/s in all,
// the LDS unit active 35 % of the time, waves waiting a third of it).
// k_wxmarch, which takes the other operators, tests every stencil's axes at
// every neighbour: 16 densities of 96^3 take 202 us there, 113 us here, 89
// repeated on one input (read and written once with the weights: 42).
#include "wstencil.h"

#include "batch.h"
#include "stencil_dev.h"

namespace gfd {

constexpr int WD_NT = 512;  // most threads of a block

template <typename T>
struct WdArgs {
    const T* in;
    T* out;
    const double* src;
    int n0, n1, n2;
    long nin;
    int tz, ty, tiles_z, tiles_y, chunks_x, xchunk, nblocks;
    double w;
    double c0[4];
    double lap[3][MAXR_FAST];   // symmetric
    double grad[3][MAXR_FAST];  // +k; -k has the opposite sign
    const double* wts[4];
    BC bc;
};

template <typename T, int R, int HM, bool RELAX>
__global__ void __launch_bounds__(WD_NT) k_wdiel(WdArgs<T> a)
{
    typedef typename ScalarOf<T>::type S;
    constexpr int U = 2 * R + 1;
    constexpr bool CPLX = IsCplx<T>::value;
    constexpr int NS = R + 2;  // ring planes: R + 1 in use, one being filled
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* lds = reinterpret_cast<T*>(smem_raw);

    const int L = xcd_remap(blockIdx.x, a.nblocks);
    const long b = L % a.nin;
    int rem = (int)(L / a.nin);
    const int zt = rem % a.tiles_z;
    rem /= a.tiles_z;
    const int yt = rem % a.tiles_y;
    const int cx = rem / a.tiles_y;

    const int tid = threadIdx.x, NT = blockDim.x;
    const int n0 = a.n0, n1 = a.n1, n2 = a.n2;
    const long ng = (long)n1 * n2 * n0;
    const unsigned plane = (unsigned)n1 * (unsigned)n2;
    const int z0 = zt * a.tz, y0 = yt * a.ty;
    const int xs = cx * a.xchunk, xe = min(xs + a.xchunk, n0);
    const int LW = a.tz + 2 * R, LSZ = (a.ty + 2 * R) * LW;
    const int buf1 = HM * NT;
    const BC& bc = a.bc;

    unsigned hoff[HM];
    bool hph[HM];
    double2 hf[HM];
#pragma unroll
    for (int m = 0; m < HM; m++) {
        const int e = tid + m * NT;
        hoff[m] = BXM_OOB;
        hph[m] = false;
        hf[m] = make_double2(1.0, 0.0);
        if (e < LSZ) {
            const int row = e / LW;
            int y = y0 + row - R, z = z0 + (e - row * LW) - R;
            if (y < n1 + R && z < n2 + R &&
                wrap_full(z, n2, bc.periodic[2], bc.phase[2][0],
                          bc.phase[2][1], hf[m], hph[m]) &&
                wrap_full(y, n1, bc.periodic[1], bc.phase[1][0],
                          bc.phase[1][1], hf[m], hph[m]))
                hoff[m] = (unsigned)(y * n2 + z) * (unsigned)sizeof(T);
        }
    }
    const int tr = tid / a.tz, tc = tid - tr * a.tz;
    const bool on = tr < a.ty && y0 + tr < n1 && z0 + tc < n2;
    const int lown = (min(tr, a.ty - 1) + R) * LW + tc + R;
    const unsigned oidx = (unsigned)((y0 + tr) * n2 + z0 + tc);
    const unsigned ooff = on ? oidx * (unsigned)sizeof(T) : BXM_OOB;
    const unsigned woff = on ? oidx * 8u : BXM_OOB;

    auto plane_at = [&](const void* base, int x, unsigned es, bool ok) {
        const unsigned pb = plane * es;
        return brsrc((const char*)base + (unsigned long)pb * (unsigned)x,
                     ok ? pb : 0u);
    };
    const void* gin = a.in + b * ng;
    void* gout = a.out + b * ng;
    T hv[HM];
    double2 fx = make_double2(1.0, 0.0);
    bool phx = false;
    auto ld_plane = [&](int x) {
        const bool lo = x < 0, hi = x >= n0;
        const int xw = lo ? x + n0 : hi ? x - n0 : x;
        const __amdgpu_buffer_rsrc_t r =
            plane_at(gin, xw, sizeof(T), !(lo || hi) || bc.periodic[0]);
        if constexpr (CPLX) {
            phx = lo || hi;
            fx = lo ? bc.phase[0][1] : bc.phase[0][0];
        }
#pragma unroll
        for (int m = 0; m < HM; m++) hv[m] = bload<T>(r, hoff[m]);
    };
    // weights (and right-hand side) of output plane x, the chunk's nearest
    // before and after it
    double wt[4], sv = 0.0;
    auto ld_weights = [&](int x) {
        const int xo = min(max(x, xs), xe - 1);
#pragma unroll
        for (int i = 0; i < 4; i++)
            wt[i] = bload<double>(plane_at(a.wts[i], xo, 8u, true), woff);
        if constexpr (RELAX)
            sv = bload<double>(plane_at(a.src, xo, 8u, true), woff);
    };

    T q[U];  // centre values of planes x - R .. x + R
#pragma unroll
    for (int j = 0; j < U; j++) q[j] = zero_of<T>();
    ld_plane(xs - R);
    ld_weights(xs);
    int wr = 0, rd = buf1 * 2;  // ring planes of x + R and of x
    for (int xb = xs - R; xb < xe + R; xb += U) {
        cfor<U>([&](auto uc) {
            constexpr int u = uc;
            const int xn = xb + u;      // plane staged in this step
            if (xn >= xe + R) return;
            const int x = xn - R;       // output plane
#pragma unroll
            for (int m = 0; m < HM; m++) {
                T v = hv[m];
                if constexpr (CPLX) {
                    if (hph[m]) v = scale_by<T>(v, hf[m], true);
                    if (phx) v = scale_by<T>(v, fx, true);
                }
                lds[wr + tid + m * NT] = v;
            }
            ld_plane(min(xn + 1, xe + R - 1));
            __syncthreads();
            // plane x + j in q[(u + j + U) mod U]: the newest is q[u + R]
            auto at = [&](auto j) -> T& {
                constexpr int i = (u + decltype(j)::value + U) % U;
                return q[i];
            };
            constexpr std::integral_constant<int, R> newest;
            constexpr std::integral_constant<int, 0> here;
            at(newest) = lds[wr + lown];
            const T* p = lds + rd + lown;
            T al = zero_of<T>(), ax = al, ay = al, az = al;
#pragma unroll
            for (int k = 1; k <= R; k++) {
                const T up = p[k], dn = p[-k];
                al = fmac(al, (S)a.lap[2][k - 1], up);
                al = fmac(al, (S)a.lap[2][k - 1], dn);
                az = fmac(az, (S)a.grad[2][k - 1], up);
                az = fmac(az, -(S)a.grad[2][k - 1], dn);
            }
#pragma unroll
            for (int k = 1; k <= R; k++) {
                const T up = p[k * LW], dn = p[-k * LW];
                al = fmac(al, (S)a.lap[1][k - 1], up);
                al = fmac(al, (S)a.lap[1][k - 1], dn);
                ay = fmac(ay, (S)a.grad[1][k - 1], up);
                ay = fmac(ay, -(S)a.grad[1][k - 1], dn);
            }
            cfor<R>([&](auto k0) {
                constexpr int k = k0 + 1;
                std::integral_constant<int, k> ahead;
                std::integral_constant<int, -k> behind;
                al = fmac(al, (S)a.lap[0][k - 1], at(ahead));
                al = fmac(al, (S)a.lap[0][k - 1], at(behind));
                ax = fmac(ax, (S)a.grad[0][k - 1], at(ahead));
                ax = fmac(ax, -(S)a.grad[0][k - 1], at(behind));
            });
            const T v = at(here);
            T r;
            if constexpr (RELAX) {
                double sum = wt[0] * al, coef = wt[0] * a.c0[0];
                sum = fma(wt[1], ax, sum);
                sum = fma(wt[2], ay, sum);
                sum = fma(wt[3], az, sum);
#pragma unroll
                for (int i = 1; i < 4; i++)
                    coef = fma(wt[i], a.c0[i], coef);
                r = (1.0 - a.w) * v + a.w * (sv - sum) / coef;
            } else {
                r = wt[0] * fmac(al, (S)a.c0[0], v);
                r = fmac(r, (S)wt[1], fmac(ax, (S)a.c0[1], v));
                r = fmac(r, (S)wt[2], fmac(ay, (S)a.c0[2], v));
                r = fmac(r, (S)wt[3], fmac(az, (S)a.c0[3], v));
            }
            const __amdgpu_buffer_rsrc_t ro =
                plane_at(gout, x, sizeof(T), x >= xs);
            if constexpr (sizeof(T) == 8) {
                bstore(r, ro, ooff);
            } else {
                typedef unsigned u4 __attribute__((ext_vector_type(4)));
                __builtin_amdgcn_raw_buffer_store_b128(
                    __builtin_bit_cast(u4, r), ro, (int)ooff, 0, 0);
            }
            ld_weights(x + 1);
            wr = wr == (NS - 1) * buf1 ? 0 : wr + buf1;
            rd = rd == (NS - 1) * buf1 ? 0 : rd + buf1;
        });
    }
}

// the operator as the kernel's coefficients; false: another pattern
static bool diel_pattern(const WAxis& st, double lap[3][MAXR_FAST],
                         double grad[3][MAXR_FAST])
{
    if (st.nw != 4 || st.R < 1 || st.R > 3) return false;
    for (int ax = 0; ax < 3; ax++)
        for (int k = 0; k < MAXR_FAST; k++) {
            if (!st.hasw[0][ax] || st.cp[0][ax][k] != st.cm[0][ax][k])
                return false;
            lap[ax][k] = st.cp[0][ax][k];
            for (int w = 1; w < 4; w++) {
                if ((st.hasw[w][ax] != 0) != (w == ax + 1)) return false;
                if (w == ax + 1) {
                    if (st.cp[w][ax][k] != -st.cm[w][ax][k]) return false;
                    grad[ax][k] = st.cp[w][ax][k];
                }
            }
        }
    return true;
}

template <typename T, int R, int HM, bool RELAX>
static int wd_launch(const WdArgs<T>& a, int threads, hipStream_t s)
{
    const size_t shm = (size_t)(R + 2) * HM * threads * sizeof(T);
    if (shm > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(
            (const void*)k_wdiel<T, R, HM, RELAX>,
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            set_error("dielectric march: %zu bytes of LDS not available "
                      "(%s)",
                      shm, hipGetErrorString(e));
            return ENOTSUP_;
        }
    }
    hipLaunchKernelGGL((k_wdiel<T, R, HM, RELAX>), dim3(a.nblocks),
                       dim3(threads), shm, s, a);
    GFD_LAUNCH_CHECK();
    return OK;
}

template <typename T, bool RELAX>
static int wd_run(const WAxis& st, const int n[3], const BC& bc,
                  const void* in, void* out, const double* src, long nin,
                  double w, hipStream_t s)
{
    WdArgs<T> a;
    if (!diel_pattern(st, a.lap, a.grad)) return ENOTSUP_;
    const int R = st.R;
    if (n[0] < R || n[1] < R || n[2] < R || nin <= 0 ||
        (long)n[1] * n[2] * (long)sizeof(T) >= (1L << 31))
        return ENOTSUP_;
    a.in = (const T*)in;
    a.out = (T*)out;
    a.src = src;
    a.n0 = n[0];
    a.n1 = n[1];
    a.n2 = n[2];
    a.nin = nin;
    a.w = w;
    a.bc = bc;
    for (int i = 0; i < 4; i++) {
        a.c0[i] = st.c0[i];
        a.wts[i] = st.wts[i];
    }
    // tile: equal parts of a row of at most 64 points by the rows of 512
    // threads (256 for 16-byte data: five ring planes of 512 would take 80
    // KB); x chunks until every CU has 16 waves
    const int nt = sizeof(T) == 16 ? 256 : 512;
    const int parts = (n[2] + 63) / 64;
    a.tz = (n[2] + parts - 1) / parts;
    const int rows = std::min(nt / a.tz, n[1]);
    a.tiles_y = (n[1] + rows - 1) / rows;
    a.ty = (n[1] + a.tiles_y - 1) / a.tiles_y;
    a.tiles_z = parts;
    const int threads = (a.tz * a.ty + 63) / 64 * 64;
    const long lsz = (long)(a.tz + 2 * R) * (a.ty + 2 * R);
    if (lsz > 4L * threads) return ENOTSUP_;
    const bool two = lsz <= 2L * threads;
    const long tiles = (long)a.tiles_z * a.tiles_y * nin;
    a.chunks_x = 1;
    while (tiles * a.chunks_x * (threads / 64) < 16 * 256 &&
           n[0] / (a.chunks_x + 1) >= 2 * R)
        a.chunks_x++;
    a.xchunk = (n[0] + a.chunks_x - 1) / a.chunks_x;
    a.chunks_x = (n[0] + a.xchunk - 1) / a.xchunk;
    const long nb = tiles * a.chunks_x;
    if (nb > 0x7fffffffL) return ENOTSUP_;
    a.nblocks = (int)nb;
    switch (R) {
    case 1: return two ? wd_launch<T, 1, 2, RELAX>(a, threads, s) : wd_launch<T, 1, 4, RELAX>(a, threads, s);
    case 2: return two ? wd_launch<T, 2, 2, RELAX>(a, threads, s) : wd_launch<T, 2, 4, RELAX>(a, threads, s);
    case 3: return two ? wd_launch<T, 3, 2, RELAX>(a, threads, s) : wd_launch<T, 3, 4, RELAX>(a, threads, s);
    }
    return ENOTSUP_;
}

int launch_wdielectric(const WAxis& st, int real, const int n[3],
                       const BC& bc, const void* in, void* out,
                       const double* src, long nin, double w, bool relax,
                       hipStream_t s)
{
    if (relax)
        return real ? wd_run<double, true>(st, n, bc, in, out, src, nin, w, s)
                    : ENOTSUP_;
    return real ? wd_run<double, false>(st, n, bc, in, out, src, nin, w, s)
                : wd_run<double2, false>(st, n, bc, in, out, src, nin, w, s);
}

}  // namespace gfd
