// Direction stencils (dirmarch.h): recognition, tile choice and dispatch.
#include "dirmarch.h"

#include <algorithm>
#include <atomic>
#include <cstdlib>

namespace gfd {

bool dir_stencil(int P, const double* coef, const int* off, DirStencil& d)
{
    d = DirStencil{};
    d.in[0].dz = 1;
    d.in[1].dy = 1;
    int ncentre = 0;
    for (int q = 0; q < P; q++) {
        const int* o = off + 3 * q;
        const int k = std::max({std::abs(o[0]), std::abs(o[1]),
                                std::abs(o[2])});
        if (k == 0) {
            if (++ncentre > 1) return false;
            continue;
        }
        if (k > MAXR_FAST) return false;
        int v[3];
        for (int c = 0; c < 3; c++) {
            if (o[c] % k != 0) return false;
            v[c] = o[c] / k;
        }
        // the sense in which the first nonzero component is positive
        int sg = 1;
        for (int c = 2; c >= 0; c--)
            if (v[c] != 0) sg = v[c];
        for (int c = 0; c < 3; c++) v[c] *= sg;
        DirLine* line = nullptr;
        if (v[0] != 0 && v[1] == 0 && v[2] == 0) {
            line = &d.x;
        } else {
            DirLine* set = v[0] ? d.mix : d.in;
            int& n = v[0] ? d.nm : d.ni;
            const int most = v[0] ? DM_NM : DM_NI;
            for (int i = 0; i < n && !line; i++)
                if (set[i].dy == v[1] && set[i].dz == v[2]) line = set + i;
            if (!line) {
                if (n == most) return false;
                line = set + n;
                line->dy = v[1];
                line->dz = v[2];
                n++;
            }
        }
        const unsigned bit = 1u << (k - 1 + (sg > 0 ? 0 : MAXR_FAST));
        if (line->has & bit) return false;
        line->has |= bit;
        (sg > 0 ? line->p : line->m)[k - 1] = coef[q];
        d.R = std::max(d.R, k);
    }
    const unsigned side = (1u << d.R) - 1, all = side | side << MAXR_FAST;
    auto mark = [&](DirLine& l) {
        l.on = !l.has ? DIR_NONE : l.has == all ? DIR_ALL : DIR_SOME;
        d.some |= l.on == DIR_SOME;
    };
    mark(d.x);
    for (DirLine& l : d.in) mark(l);
    for (DirLine& l : d.mix) mark(l);
    if (!d.some && d.ni == 2 && d.nm == 0 &&
        (d.x.on != 0) + (d.in[0].on != 0) + (d.in[1].on != 0) == 1)
        d.line = d.x.on ? 0 : d.in[1].on ? 1 : 2;
    auto full = [](const DirLine& l) {
        return l.on == DIR_ALL && std::equal(l.p, l.p + MAXR_FAST, l.m);
    };
    d.full = full(d.x) && std::all_of(d.in, d.in + d.ni, full) &&
             std::all_of(d.mix, d.mix + d.nm, full);
    return d.R > 0;
}

constexpr int DM_THREADS = 512;

static std::mutex g_dm_mu;
static bool g_dm_override = false;
static DirTile g_dm_tile;

void dirmarch_set_tile(const XmTile* t)
{
    std::lock_guard<std::mutex> lk(g_dm_mu);
    g_dm_override = t != nullptr;
    if (t) {
        const int ty = t->nseg * t->py;
        g_dm_tile = DirTile{t->tz, ty, t->xchunk,
                            (t->tz * ty + 63) / 64 * 64};
    }
}

// Tile (equal parts of a row by as many rows as 512 or 256 threads hold,
// the rows split evenly) and x chunk with the least estimated time:
//   planes per block (every chunk stages 2R planes more)
//   x waves of all blocks of one CU x (1 + 0.12 per staged element)
//   x (1 + 4 / resident waves per CU): too few do not hide the latency
//   x (1 + 0.2 x cache lines loaded per line of results): short rows and
//     small tiles load partial lines and more halo.
// The weights fit measured sweeps (48 c128 grids of 128^3: 64 x 8 threads
// 703 us, 128 x 4 with 4 staged elements 795, 32 x 8 802; 40 f64 grids of
// 87x103x95: 48 x 10 in two chunks 174 us, whole x 184, 95 x 5 209; 24 c128
// grids of 60x60x84, hexagonal, repeated on one input: 28 x 9 in two chunks
// 55 us, whole x 58, in four 64).
// pad: blocks of more threads than tile points, enough to stage the halo.
static bool dm_search(const DirStencil& d, int dtype, const int n[3],
                      long nin, int epi, bool pad, DirTile& best)
{
    const int R = d.R;
    const DirHalo h = dir_halo(R, dir_line(d, dtype, epi));
    // waves a CU holds: two blocks of 8 at the 86 registers of complex FP64
    // at R = 3
    const int hold = dtype == 1 && R > 1 ? 16 : 32;
    double least = 1e300;
    for (int parts = 1; parts <= n[2]; parts++) {
        DirTile t;
        t.tz = (n[2] + parts - 1) / parts;
        if (t.tz > DM_THREADS) continue;
        if (t.tz < 16 && parts > 1) break;
        for (int nt = DM_THREADS; nt >= DM_THREADS / 2; nt /= 2) {
            if (t.tz > nt) break;
            const int rows = std::min(nt / t.tz, n[1]);
            const int nr = (n[1] + rows - 1) / rows;
            t.ty = (n[1] + nr - 1) / nr;
            t.threads = (t.tz * t.ty + 63) / 64 * 64;
            const long lsz = (long)(t.tz + 2 * h.z) * (t.ty + 2 * h.y);
            if (pad) t.threads = std::max(t.threads,
                                          (int)((lsz + 255) / 256 * 64));
            if (lsz > 4L * t.threads || t.threads > DM_THREADS) continue;
            const int hm = lsz <= t.threads ? 1 : lsz <= 2L * t.threads ? 2
                                                                        : 4;
            const int waves = t.threads / 64;
            const int es = dtype == 1 ? 16 : dtype == 2 ? 4 : 8;
            const double lines = (t.ty + 2 * h.y) *
                                 ((t.tz + 2 * h.z) * es / 128.0 + 1.0) /
                                 (t.tz * t.ty * es / 128.0);
            const long tiles = (long)parts * nr * nin;
            for (int chunks = 1; chunks <= n[0]; chunks++) {
                t.xchunk = (n[0] + chunks - 1) / chunks;
                const long blocks =
                    tiles * ((n[0] + t.xchunk - 1) / t.xchunk);
                const long per = (blocks + 255) / 256;
                // fewer than four planes: only where half the CUs are idle
                // (one c128 grid of 23^3, R = 4: 11.6 -> 10.2 us)
                if (4 * chunks > n[0] && chunks > 1 &&
                    (blocks > 128 || h.x == 0))
                    break;
                const double resident =
                    std::min<long>(per, std::max(1, hold / waves)) * waves;
                const double cost = (double)(t.xchunk + 2 * h.x) * per * waves *
                                    (1.0 + 0.12 * hm) *
                                    (1.0 + 4.0 / resident) *
                                    (1.0 + 0.2 * lines);
                if (cost < least) {
                    least = cost;
                    best = t;
                }
                if (per * waves > 4 * hold) break;
            }
        }
    }
    return least < 1e300;
}

static std::atomic<long> g_dm_searches{0};

DirTile dir_tile(const DirStencil& d, int dtype, const int n[3], long nin,
                 int epi)
{
    g_dm_searches++;
    DirTile t{};
    // At R = 4 the halo of a few short rows (4 of 14 to 16 points, 5 of 12)
    // is more than four points for each thread of their only tile.
    if (!dm_search(d, dtype, n, nin, epi, false, t))
        dm_search(d, dtype, n, nin, epi, true, t);
    return t;
}

DirTile DirTiles::get(const DirStencil& d, int dtype, const int n[3],
                      long nin, int epi)
{
    const int line = dir_line(d, dtype, epi);
    std::lock_guard<std::mutex> lk(mu);
    for (int i = 0; i < used; i++)
        if (e[i].nin == nin && e[i].dtype == dtype && e[i].line == line)
            return e[i].t;
    Entry& x = e[next];
    x = Entry{dtype, line, nin, dir_tile(d, dtype, n, nin, epi)};
    next = (next + 1) % MOST;
    used = std::max(used, next ? next : MOST);
    return x.t;
}

bool dirmarch_fits(const DirStencil& d, int dtype, const int n[3], int epi)
{
    if (d.R < 1 || d.R > MAXR_FAST ||
        (d.R > DM_RSKEW && (d.ni > 2 || d.nm > 0)))
        return false;
    if (n[0] < d.R || n[1] < d.R || n[2] < d.R) return false;
    const long es = dtype == 1 ? 16 : 8;  // widest operand of a pass
    if (dtype == 3 ? (long)n[1] * n[2] * 16 >= (1L << 31)
                   : (long)n[1] * n[2] * es >= (1L << 31))
        return false;
    if (epi == EPI_RELAX && (dtype == 1 || dtype == 3)) return false;
    if (epi == EPI_POT && dtype > 1) return false;
    if (epi == EPI_UPDW && dtype < 2) return false;
    if (epi == EPI_RESN && dtype != 0) return false;
    return true;
}

long dirmarch_max_blocks(const DirStencil& d, DirTiles& tiles, int dtype,
                         const int n[3], long nin)
{
    if (d.R < 1 || std::min({n[0], n[1], n[2]}) < d.R) return 0;
    const DirTile t = tiles.get(d, dtype, n, nin, EPI_RESID);
    return (long)ceil_div(n[2], t.tz) * ceil_div(n[1], t.ty) *
           ceil_div(n[0], t.xchunk) * nin;
}

int launch_dirmarch(const DirStencil& d, DirTiles& tiles, int dtype,
                    const int n[3], const BC& bc, const void* in, void* out,
                    long nin, int epi, const EpiArgs& ea, hipStream_t s,
                    int* nblocks_out)
{
    DirTile t = tiles.get(d, dtype, n, nin, epi);
    if (!ea.partial) {
        std::lock_guard<std::mutex> lk(g_dm_mu);
        const DirTile& o = g_dm_tile;
        if (g_dm_override && o.threads <= DM_THREADS &&
            (o.tz + 2 * d.R) * (o.ty + 2 * d.R) <= 4 * o.threads)
            t = o;
    }
    switch (dtype) {
    case 0: return dirmarch_f64(d, t, n, bc, in, out, nin, epi, ea, s, nblocks_out);
    case 1: return dirmarch_c128(d, t, n, bc, in, out, nin, epi, ea, s, nblocks_out);
    case 2: return dirmarch_f32(d, t, n, bc, in, out, nin, epi, ea, s, nblocks_out);
    case 3: return dirmarch_c64(d, t, n, bc, in, out, nin, epi, ea, s, nblocks_out);
    }
    set_error("direction march: unsupported data type %d", dtype);
    return ENOTSUP_;
}

}  // namespace gfd

extern "C" int gfd_march_tile(int npoints, const double* coefs,
                              const int* offsets, const int n[3], int dtype,
                              long nin, int plain, int tile[4])
{
    if (!coefs || !offsets || !n || !tile || npoints < 1 || nin < 1 ||
        dtype < 0 || dtype > 3 || n[0] < 1 || n[1] < 1 || n[2] < 1) {
        gfd::set_error("gfd_march_tile: bad arguments");
        return gfd::EINVAL_;
    }
    gfd::DirStencil d;
    if (!gfd::dir_stencil(npoints, coefs, offsets, d) ||
        !gfd::dirmarch_fits(d, dtype, n, gfd::EPI_PLAIN)) {
        gfd::set_error("gfd_march_tile: not for the direction march");
        return gfd::ENOTSUP_;
    }
    const gfd::DirTile t =
        gfd::dir_tile(d, dtype, n, nin, plain ? gfd::EPI_PLAIN
                                              : gfd::EPI_RESID);
    tile[0] = t.tz;
    tile[1] = t.ty;
    tile[2] = t.xchunk;
    tile[3] = t.threads;
    return gfd::OK;
}

extern "C" long gfd_march_tile_searches(void)
{
    return gfd::g_dm_searches;
}
