// Temporally blocked smoothing of the coarse multigrid levels.
//
// A level below the finest (7-point stencil) costs a V-cycle up to ten
// launches -- sweeps, residual, restriction, interpolation, sweeps -- each a
// few microseconds of latency for arrays that the caches hold.  Here each
// half of its visit is one launch: a block takes an 8 x 8 x 8 tile with a
// halo as wide as the work needs (one point per sweep, and one for the
// residual), and recomputes the halo instead of exchanging it.
//
//   down: sweeps from zero (the first is the scaled right-hand side), the
//         residual, its restriction to the tile's 4 x 4 x 4 coarse points
//   up:   the interpolated correction, then the sweeps
//
// A thread owns one x column of the extended tile: iterate and right-hand
// side in registers, the four in-plane neighbours from LDS, values beyond
// the sweep's valid range left as they are (they spread one point inward
// per sweep, which is what the halo is for).  Points outside a zero boundary
// stay zero; periodic axes wrap on load.
//
// What bounds it: one load latency and two barriers per sweep.  FP64 24^3, 4
// sweeps each way: down 10 us (6 launches before, about 45 us with their
// gaps), up 14 us (5 launches, 40 us); FP32 96^3, 3 and 4 sweeps: 16 and 29
// us (separate launches 45 and 50).  48^3 FP64 solve 2.06 -> 1.62 ms, 192^3
// mixed solve 5.60 -> 4.52 ms, twelve uneven grids batched 8.24 -> 6.88 ms.
#include "tsmooth.h"

#include <algorithm>
#include <atomic>

#include "stencil_dev.h"

namespace gfd {

template <typename T>
struct TsArgs {
    const TsGrid* g;
    int G;
    const T* rhs;
    const T* e_in;
    const T* c;
    T* e_out;
    T* rhs_c;
};

// index along an axis: wrapped, or -1 outside a zero boundary
__device__ inline int ts_wrap(int i, int n, int periodic)
{
    if (i >= 0 && i < n) return i;
    if (!periodic) return -1;
    while (i < 0) i += n;
    while (i >= n) i -= n;
    return i;
}

constexpr int ts_halo(int S, bool up) { return up ? S : S + 1; }
constexpr int ts_side(int S, bool up) { return TS_B + 2 * ts_halo(S, up); }
constexpr int ts_threads(int S, bool up)
{
    return (ts_side(S, up) * ts_side(S, up) + 63) / 64 * 64;
}

template <typename T, int S, bool UP>
__global__ void __launch_bounds__(ts_threads(S, UP)) k_tsmooth(TsArgs<T> a)
{
    typedef typename ScalarOf<T>::type R;
    constexpr int H = ts_halo(S, UP), D = ts_side(S, UP);
    constexpr int DC = D / 2 + 2;  // coarse points under the extended tile
    __shared__ T E[D * D * D];
    __shared__ T C[UP ? DC * DC * DC : 1];
    // the tile's grid: the last one whose first tile is not past it
    int lo = 0, hi = a.G - 1;
    const int tile = blockIdx.x;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.g[mid].tile0 <= tile) lo = mid;
        else hi = mid - 1;
    }
    const TsGrid g = a.g[lo];
    int lt = tile - g.tile0;
    int tb[3];
    tb[2] = lt % g.tiles[2];
    lt /= g.tiles[2];
    tb[1] = lt % g.tiles[1];
    tb[0] = lt / g.tiles[1];
    const int nt = ts_threads(S, UP), t = threadIdx.x;
    const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
    const int x0 = tb[0] * TS_B - H;
    // own column of the extended tile
    const int y = t / D, z = t - y * D;
    const int gy = tb[1] * TS_B - H + y, gz = tb[2] * TS_B - H + z;
    const int yw = ts_wrap(gy, n1, g.periodic[1]);
    const int zw = ts_wrap(gz, n2, g.periodic[2]);
    const bool col = y < D && yw >= 0 && zw >= 0;
    const int own = col ? yw * n2 + zw : 0;
    const long plane = (long)n1 * n2;

    T r[D], e[D];
    const T* rl = a.rhs + g.off;
    const T* ei = UP ? a.e_in + g.off : rl;
    unsigned inside = 0;  // bit i: plane x0 + i is inside the grid
    cfor<D>([&](auto i) {
        const int x = ts_wrap(x0 + i, n0, g.periodic[0]);
        if (x >= 0) inside |= 1u << i;
        const long p = (long)x * plane + own;
        r[i] = col && x >= 0 ? rl[p] : (T)0;
        if constexpr (UP) e[i] = col && x >= 0 ? ei[p] : (T)0;
    });
    const R wc = (R)(g.w / g.c0), w1 = (R)(1.0 - g.w), c0 = (R)g.c0;
    if constexpr (UP) {
        // coarse points under the tile
        int cb[3];
#pragma unroll
        for (int d = 0; d < 3; d++)
            cb[d] = ((tb[d] * TS_B - H + g.iskip0[d]) >> 1) + g.ioff[d];
        const T* cl = a.c + g.offc;
        for (int p = t; p < DC * DC * DC; p += nt) {
            const int cx = ts_wrap(cb[0] + p / (DC * DC), g.nc[0],
                                   g.periodic[0]);
            const int cy = ts_wrap(cb[1] + p / DC % DC, g.nc[1],
                                   g.periodic[1]);
            const int cz = ts_wrap(cb[2] + p % DC, g.nc[2], g.periodic[2]);
            C[p] = cx >= 0 && cy >= 0 && cz >= 0
                       ? cl[((long)cx * g.nc[1] + cy) * g.nc[2] + cz]
                       : (T)0;
        }
        __syncthreads();
        if (col) {
            const int q1 = gy + g.iskip0[1], q2 = gz + g.iskip0[2];
            const int c1 = (q1 >> 1) + g.ioff[1] - cb[1];
            const int c2 = (q2 >> 1) + g.ioff[2] - cb[2];
            const bool h1 = q1 & 1, h2 = q2 & 1;
            // the column's value at each coarse plane under it
            T v[DC];
            cfor<DC>([&](auto j) {
                const T* p = C + (j * DC + c1) * DC + c2;
                T v0 = p[0];
                if (h2) v0 = (R)0.5 * (v0 + p[1]);
                if (h1) {
                    T v1 = p[DC];
                    if (h2) v1 = (R)0.5 * (v1 + p[DC + 1]);
                    v0 = (R)0.5 * (v0 + v1);
                }
                v[j] = v0;
            });
            // plane i lies on coarse plane (i + odd) / 2 or half way on
            auto correct = [&](auto odd) {
                cfor<D>([&](auto i) {
                    constexpr int q = i + odd, j = q / 2;
                    T c = v[j];
                    if constexpr (q % 2) c = (R)0.5 * (c + v[j + 1]);
                    if (inside >> i & 1u) e[i] = e[i] - c;
                });
            };
            if ((x0 + g.iskip0[0]) & 1)
                correct(std::integral_constant<int, 1>{});
            else
                correct(std::integral_constant<int, 0>{});
        }
    } else {
        cfor<D>([&](auto i) { e[i] = wc * r[i]; });
    }
    T* E0 = E + y * D + z;
    const bool in = y < D;
    if (in)
        cfor<D>([&](auto i) { E0[i * D * D] = e[i]; });
    __syncthreads();

    const R cpx = (R)g.cp[0], cmx = (R)g.cm[0], cpy = (R)g.cp[1],
            cmy = (R)g.cm[1], cpz = (R)g.cp[2], cmz = (R)g.cm[2];
    // f(i, acc) for the points of the column at least LO from the extended
    // tile's faces and inside the grid (acc: off-centre terms, z, y, x)
    auto pass = [&](auto lo_, auto&& f) {
        constexpr int LO = lo_;
        if (!col || y < LO || y >= D - LO || z < LO || z >= D - LO) return;
        T below = e[LO - 1];
        cfor<D - 2 * LO>([&](auto i_) {
            constexpr int i = i_ + LO;
            const T* p = E0 + i * D * D;
            T acc = (T)0;
            acc = fmac(acc, cpz, p[1]);
            acc = fmac(acc, cmz, p[-1]);
            acc = fmac(acc, cpy, p[D]);
            acc = fmac(acc, cmy, p[-D]);
            acc = fmac(acc, cpx, e[i + 1]);
            acc = fmac(acc, cmx, below);
            below = e[i];
            if (inside >> i & 1u) f(std::integral_constant<int, i>{}, acc);
        });
    };
    // the last sweep of an up pass stays in registers
    constexpr int FIRST = UP ? 1 : 2;
    cfor<S - FIRST + 1>([&](auto k_) {
        constexpr int k = k_ + FIRST;
        constexpr int LO = UP ? k : k - 1;
        std::integral_constant<int, LO> lo_;
        pass(lo_, [&](auto i, T acc) {
            e[i] = fmac(w1 * e[i], wc, r[i] - acc);
        });
        if constexpr (!UP || k < S) {
            __syncthreads();
            if (col && y >= LO && y < D - LO && z >= LO && z < D - LO)
                cfor<D - 2 * LO>([&](auto i_) {
                    constexpr int i = i_ + LO;
                    E0[i * D * D] = e[i];
                });
            __syncthreads();
        }
    });
    // the tile's own points
    if (y >= H && y < H + TS_B && z >= H && z < H + TS_B && gy < n1 &&
        gz < n2) {
        T* o = a.e_out + g.off + (long)gy * n2 + gz;
        cfor<TS_B>([&](auto i_) {
            constexpr int i = i_ + H;
            if (x0 + i < n0) o[(long)(x0 + i) * plane] = e[i];
        });
    }
    if constexpr (!UP) {
        // residual (zero outside the grid) one point beyond the tile
        std::integral_constant<int, S> lo_;
        T q[D];
        cfor<D>([&](auto i) { q[i] = (T)0; });
        pass(lo_, [&](auto i, T acc) {
            q[i] = fmac(acc, c0, e[i]) - r[i];
        });
        __syncthreads();
        if (in && y >= S && y < D - S && z >= S && z < D - S)
            cfor<D - 2 * S>([&](auto i_) {
                constexpr int i = i_ + S;
                E0[i * D * D] = q[i];
            });
        __syncthreads();
        if (t < 64) {
            const int cz = t & 3, cy = t >> 2 & 3, cx = t >> 4;
            const int oz = tb[2] * 4 + cz, oy = tb[1] * 4 + cy,
                      ox = tb[0] * 4 + cx;
            if (ox < g.nc[0] && oy < g.nc[1] && oz < g.nc[2]) {
                const T* p = E + ((H + 2 * cx + g.roff[0]) * D + H + 2 * cy +
                                  g.roff[1]) * D + H + 2 * cz + g.roff[2];
                T px[3];
#pragma unroll
                for (int dx = 0; dx < 3; dx++) {
                    T py[3];
#pragma unroll
                    for (int dy = 0; dy < 3; dy++) {
                        const T* w = p + ((dx - 1) * D + dy - 1) * D;
                        py[dy] = (R)0.5 * fmac(w[0], (R)0.5, w[1] + w[-1]);
                    }
                    px[dx] = (R)0.5 * fmac(py[1], (R)0.5, py[2] + py[0]);
                }
                a.rhs_c[g.offc + ((long)ox * g.nc[1] + oy) * g.nc[2] + oz] =
                    (R)0.5 * fmac(px[1], (R)0.5, px[2] + px[0]);
            }
        }
    }
}

static std::atomic<bool> g_ts{true};

void ts_set_enabled(bool on) { g_ts = on; }
bool ts_enabled() { return g_ts; }

int ts_tiles(TsGrid& g)
{
    int total = 1;
    for (int c = 0; c < 3; c++) {
        g.tiles[c] = (g.n[c] + TS_B - 1) / TS_B;
        total *= g.tiles[c];
    }
    return total;
}

template <typename T, bool UP>
static int ts_launch(const TsArgs<T>& a, long ntiles, int sweeps,
                     hipStream_t s)
{
    if (ntiles <= 0) return OK;
    if (ntiles > 0x7fffffffL) {
        set_error("blocked smoothing: too many tiles (%ld)", ntiles);
        return ENOTSUP_;
    }
#define GFD_TS(S)                                                           \
    case S:                                                                 \
        hipLaunchKernelGGL((k_tsmooth<T, S, UP>), dim3((unsigned)ntiles),   \
                           dim3(ts_threads(S, UP)), 0, s, a);               \
        break
    switch (sweeps) {
        GFD_TS(1);
        GFD_TS(2);
        GFD_TS(3);
        GFD_TS(4);
    default:
        set_error("blocked smoothing: %d sweeps", sweeps);
        return ENOTSUP_;
    }
#undef GFD_TS
    GFD_LAUNCH_CHECK();
    return OK;
}

int launch_ts_down(const TsGrid* d, int G, long ntiles, int dtype, int sweeps,
                   const void* rhs, void* e, void* rhs_c, hipStream_t s)
{
    if (dtype == 2)
        return ts_launch<float, false>({d, G, (const float*)rhs, nullptr,
                                        nullptr, (float*)e, (float*)rhs_c},
                                       ntiles, sweeps, s);
    return ts_launch<double, false>({d, G, (const double*)rhs, nullptr,
                                     nullptr, (double*)e, (double*)rhs_c},
                                    ntiles, sweeps, s);
}

int launch_ts_up(const TsGrid* d, int G, long ntiles, int dtype, int sweeps,
                 const void* rhs, const void* e, const void* c, void* e_out,
                 hipStream_t s)
{
    if (dtype == 2)
        return ts_launch<float, true>({d, G, (const float*)rhs,
                                       (const float*)e, (const float*)c,
                                       (float*)e_out, nullptr},
                                      ntiles, sweeps, s);
    return ts_launch<double, true>({d, G, (const double*)rhs,
                                    (const double*)e, (const double*)c,
                                    (double*)e_out, nullptr},
                                   ntiles, sweeps, s);
}

}  // namespace gfd
