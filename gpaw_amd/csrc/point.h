// Axis stencils on few real points (point.hip).
#pragma once

#include "stencil.h"

namespace gfd {

// Most points (all grids) for one point per thread, FP64 and FP32 data.
// Graph replays of the nn=3 Laplacian, marching against this: FP64 48^3 8.1
// / 3.7 us, 64^3 8.3 / 5.4, 80^3 9.0 / 8.1, 96^3 10.3 / 11.8, 8 x 48^3 9.8 /
// 10.9; nn=1 96^3 6.8 / 6.6.  Whole solves with FP32 sweeps: 96^3 2.58 /
// 2.28 ms, 128^3 3.00 / 3.33 ms.
constexpr double PT_MAX64 = 600e3, PT_MAX32 = 1000e3;

bool point_fits(const AxisStencil& st, int dtype, const int n[3], long nin,
                int epi);
int launch_point(const AxisStencil& st, int dtype, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out);

}  // namespace gfd
