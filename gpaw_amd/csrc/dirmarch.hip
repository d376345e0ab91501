// Direction stencils (dirmarch.h): recognition, tile choice and dispatch.
#include "dirmarch.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>

namespace gfd {

bool dir_stencil(int P, const double* coef, const int* off, DirStencil& d)
{
    d = DirStencil{};
    d.in[0].dz = 1;
    d.in[1].dy = 1;
    bool seen[1 + DM_NI + DM_NM][2 * MAXR_FAST + 1] = {};
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
        int id = -1;
        if (v[0] != 0 && v[1] == 0 && v[2] == 0) {
            line = &d.x;
            id = 0;
        } else {
            DirLine* set = v[0] ? d.mix : d.in;
            int& n = v[0] ? d.nm : d.ni;
            const int most = v[0] ? DM_NM : DM_NI;
            for (int i = 0; i < n && !line; i++)
                if (set[i].dy == v[1] && set[i].dz == v[2]) {
                    line = set + i;
                    id = 1 + i + (v[0] ? DM_NI : 0);
                }
            if (!line) {
                if (n == most) return false;
                line = set + n;
                line->dy = v[1];
                line->dz = v[2];
                id = 1 + n + (v[0] ? DM_NI : 0);
                n++;
            }
        }
        line->on = 1;
        bool& s = seen[id][MAXR_FAST + sg * k];
        if (s) return false;
        s = true;
        (sg > 0 ? line->p : line->m)[k - 1] = coef[q];
        d.R = std::max(d.R, k);
    }
    auto same = [](const DirLine& l) {
        return std::equal(l.p, l.p + MAXR_FAST, l.m);
    };
    d.sym = same(d.x);
    for (const DirLine& l : d.in) d.sym = d.sym && same(l);
    for (const DirLine& l : d.mix) d.sym = d.sym && same(l);
    return d.R > 0;
}

// largest radius of the skew forms (9 accumulators and their directions do
// not fit the registers)
constexpr int DM_RSKEW = 3;
constexpr int DM_THREADS = 512;
constexpr int DM_STAGED = 4;  // staged elements per thread

static bool tile_fits(const DirTile& t, int R)
{
    const int threads = (t.tz * t.ty + 63) / 64 * 64;
    return t.tz >= 1 && t.ty >= 1 && t.xchunk >= 1 && threads <= DM_THREADS &&
           (long)(t.tz + 2 * R) * (t.ty + 2 * R) <= (long)DM_STAGED * threads;
}

// Tile: equal parts of a row by as many rows as a block holds, the pair with
// the least work for the whole plane, counting a staged element (a load
// from L2 and an LDS write) like half a computed lane.  x chunks: whole x
// unless that leaves the chip idle; every chunk stages 2R planes more, and
// about two blocks of 512 threads are resident per CU.
static bool dm_tile(const DirStencil& d, const int n[3], long nin, DirTile& t)
{
    const int R = d.R;
#ifdef DM_PROBE
    if (const char* e = getenv("DM_TILE")) {
        if (sscanf(e, "%d,%d,%d", &t.tz, &t.ty, &t.xchunk) == 3) {
            t.xchunk = std::min(t.xchunk, n[0]);
            if (tile_fits(t, R)) return true;
        }
    }
#endif
    double best = 1e300;
    bool found = false;
    for (int parts = 1; parts <= n[2]; parts++) {
        DirTile c;
        c.tz = (n[2] + parts - 1) / parts;
        c.xchunk = n[0];
        if (c.tz > DM_THREADS) continue;
        if (c.tz < 12 && parts > 1) break;
        for (int ry = 1; ry <= n[1]; ry++) {
            c.ty = (n[1] + ry - 1) / ry;
            if (!tile_fits(c, R)) continue;
            const int threads = (c.tz * c.ty + 63) / 64 * 64;
            const double cost =
                (double)((n[2] + c.tz - 1) / c.tz) *
                ((n[1] + c.ty - 1) / c.ty) *
                (threads + 0.5 * (c.tz + 2 * R) * (c.ty + 2 * R));
            if (cost < best) {
                best = cost;
                t = c;
                found = true;
            }
        }
    }
    if (!found) return false;
    const int threads = (t.tz * t.ty + 63) / 64 * 64;
    const long tiles = (long)((n[2] + t.tz - 1) / t.tz) *
                       ((n[1] + t.ty - 1) / t.ty) * nin;
    const long resident = 256L * std::max(1, 1024 / threads);
    double least = 1e300;
    for (int chunks = 1; chunks <= std::max(1, n[0] / 4); chunks++) {
        const int xc = (n[0] + chunks - 1) / chunks;
        const long blocks = tiles * ((n[0] + xc - 1) / xc);
        const double rounds = blocks <= 8 * resident
                                  ? (double)((blocks + resident - 1) / resident)
                                  : (double)blocks / resident;
        const double cost = rounds * (xc + 2 * R);
        if (cost < least * 0.98) {
            least = cost;
            t.xchunk = xc;
        }
        if (blocks > 8 * resident) break;
    }
    return true;
}

bool dirmarch_fits(const DirStencil& d, int dtype, const int n[3], long nin,
                   int epi)
{
    if (d.R < 1 || d.R > MAXR_FAST ||
        (d.R > DM_RSKEW && (d.ni > 2 || d.nm > 0)))
        return false;
    if (n[0] < d.R || n[1] < d.R || n[2] < d.R) return false;
    const long es = dtype == 1 ? 16 : 8;  // widest operand of a pass
    if (dtype == 3 ? (long)n[1] * n[2] * 16 >= (1L << 31)
                   : (long)n[1] * n[2] * es >= (1L << 31))
        return false;
    if (!d.sym && epi != EPI_PLAIN) return false;
    if (epi == EPI_RELAX && (dtype == 1 || dtype == 3)) return false;
    if (epi == EPI_POT && dtype > 1) return false;
    if (epi == EPI_UPDW && dtype < 2) return false;
    if (epi == EPI_RESN && dtype != 0) return false;
    DirTile t;
    return dm_tile(d, n, nin, t);
}

long dirmarch_max_blocks(const DirStencil& d, int dtype, const int n[3],
                         long nin)
{
    (void)dtype;
    DirTile t;
    if (d.R < 1 || !dm_tile(d, n, nin, t)) return 0;
    return (long)ceil_div(n[2], t.tz) * ceil_div(n[1], t.ty) *
           ceil_div(n[0], t.xchunk) * nin;
}

int launch_dirmarch(const DirStencil& d, int dtype, const int n[3],
                    const BC& bc, const void* in, void* out, long nin,
                    int epi, const EpiArgs& ea, hipStream_t s,
                    int* nblocks_out)
{
    DirTile t;
    if (!dm_tile(d, n, nin, t)) {
        set_error("direction march: no tile fits this grid");
        return ENOTSUP_;
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
