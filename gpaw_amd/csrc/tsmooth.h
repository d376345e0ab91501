// Temporally blocked smoothing of the coarse multigrid levels (tsmooth.hip).
#pragma once

#include "gfd_common.h"

namespace gfd {

constexpr int TS_B = 8;       // fine points of a tile per axis
constexpr int TS_MAXS = 4;    // sweeps of one launch

// One grid's level: a 7-point stencil, its transfers to and from the next
// coarser level, and its place in the level's arrays.
struct TsGrid {
    int n[3], nc[3], periodic[3];
    int roff[3];             // restriction: first centre per axis (0 or 1)
    int ioff[3], iskip0[3];  // interpolation back
    int tiles[3], tile0;
    long off, offc;
    double c0, w;
    double cp[3], cm[3];
};

// tiles[] of a grid from n; returns their number
int ts_tiles(TsGrid& g);

// Most points of a level (all grids of a batch) for which the blocked half
// cycles are used: beyond, the recomputed halos cost more than the launches
// (a level of 0.9 million points in 12 grids: the batched solve 17 % faster;
// 1.8 million in 24 grids: 11 %; a level of 5 million would break even)
constexpr long TS_PTS = 2000000;

// Off: every level keeps its separate launches (tuning key "tsmooth").
void ts_set_enabled(bool on);
bool ts_enabled();

// `sweeps` Jacobi sweeps from zero for A e = rhs, then the restricted
// residual: rhs_c = R (A e - rhs).  dtype 0 f64, 2 f32.
int launch_ts_down(const TsGrid* d, int G, long ntiles, int dtype, int sweeps,
                   const void* rhs, void* e, void* rhs_c, hipStream_t s);
// e_out = `sweeps` Jacobi sweeps from e - I c (e_out not e).
int launch_ts_up(const TsGrid* d, int G, long ntiles, int dtype, int sweeps,
                 const void* rhs, const void* e, const void* c, void* e_out,
                 hipStream_t s);

}  // namespace gfd
