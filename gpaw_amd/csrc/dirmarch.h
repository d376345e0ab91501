// Stencils made of straight lines of points through the centre (axis
// stencils, the Laplacians and gradients of skew cells), marching along x.
#pragma once

#include <mutex>

#include "stencil.h"

namespace gfd {

constexpr int DM_NI = 3;  // in-plane directions: (0, 1), (1, 0) and one more
constexpr int DM_NM = 4;  // directions (1, dy, dz) off the x axis
// largest radius the skew forms are built for.  (Radius 4 would fit: the
// hexagonal Laplacian compiles to 103 registers in complex FP64 and no
// scratch.  It is not built; those cells run on k_general.)
constexpr int DM_RSKEW = 3;

// What a stencil has on a line: no points, points at every step 1..R on both
// sides, or some of them (bits k - 1 of `has` for +k, MAXR_FAST + k - 1 for
// -k).  A point that is not there is not read: multiplied by zero it would
// turn an infinity into NaN.
enum DirOn : int { DIR_NONE = 0, DIR_ALL = 1, DIR_SOME = 2 };

// in(x + k d) has coefficient p[k - 1], in(x - k d) m[k - 1], k = 1..R
struct DirLine {
    int on;      // DirOn
    unsigned has;
    int dy, dz;
    double p[MAXR_FAST], m[MAXR_FAST];
};

struct DirStencil {
    int R = 0;
    int ni = 2, nm = 0;  // in-plane / mixed directions
    int full = 0;  // x and the ni, nm directions all DIR_ALL, p[k] = m[k]
    int some = 0;  // one of them is DIR_SOME
    int line = -1; // the axis of a stencil of one DIR_ALL axis line
    DirLine x, in[DM_NI], mix[DM_NM];
};

// The direction form of P points (offsets as triples); false when a point is
// not a multiple of a direction with components -1, 0, 1, is given twice,
// lies beyond MAXR_FAST steps, or more directions are needed.
bool dir_stencil(int P, const double* coef, const int* off, DirStencil& d);

// Tile in place of the estimated one (tuning key "xm_tile"; rows nseg x py),
// where it fits and the pass sums no norm (its buffer is sized for the
// estimated tile); nullptr clears.
void dirmarch_set_tile(const XmTile* t);

// Columns and rows of a tile, planes of an x chunk, threads of a block (one
// per tile point, or more where the tile with its halo needs them to stage
// it at four points each).
struct DirTile {
    int tz, ty, xchunk, threads;
};

// Widths of what a block stages beyond its points along y and z, and of the
// planes it marches through beyond its chunk.
struct DirHalo {
    int x, y, z;
};

// A plain FP64 pass of a stencil on one axis reads along that axis only (the
// other epilogues, and FP32 data, which has no gradients, run the general
// form).
constexpr DirHalo dir_halo(int R, int line)
{
    return {line < 1 ? R : 0, line < 0 || line == 1 ? R : 0,
            line < 0 || line == 2 ? R : 0};
}
inline int dir_line(const DirStencil& d, int dtype, int epi)
{
    return epi == EPI_PLAIN && dtype < 2 ? d.line : -1;
}

// The tile with the least estimated time; every grid of sides >= R has one.
// A search of 1 to 11 us on the host (8 f64 grids of 48^3, one c128 grid of
// 160^3), as long as the kernels of small grids run.
DirTile dir_tile(const DirStencil& d, int dtype, const int n[3], long nin,
                 int epi);

// The tiles one operator has used, by data type, batch and halo: looked up on
// each launch, from any thread.  The oldest of them makes room for a new one.
class DirTiles {
public:
    DirTile get(const DirStencil& d, int dtype, const int n[3], long nin,
                int epi);

private:
    struct Entry {
        int dtype, line;
        long nin;
        DirTile t;
    };
    static constexpr int MOST = 16;
    std::mutex mu;
    Entry e[MOST];
    int used = 0, next = 0;
};

// Whether k_dirmarch takes this pass.
bool dirmarch_fits(const DirStencil& d, int dtype, const int n[3], int epi);
long dirmarch_max_blocks(const DirStencil& d, DirTiles& tiles, int dtype,
                         const int n[3], long nin);
int launch_dirmarch(const DirStencil& d, DirTiles& tiles, int dtype,
                    const int n[3], const BC& bc, const void* in, void* out,
                    long nin, int epi, const EpiArgs& ea, hipStream_t s,
                    int* nblocks_out);

int dirmarch_f64(const DirStencil& d, const DirTile& t, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out);
int dirmarch_c128(const DirStencil& d, const DirTile& t, const int n[3],
                  const BC& bc, const void* in, void* out, long nin, int epi,
                  const EpiArgs& ea, hipStream_t s, int* nblocks_out);
int dirmarch_f32(const DirStencil& d, const DirTile& t, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out);
int dirmarch_c64(const DirStencil& d, const DirTile& t, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out);

}  // namespace gfd
