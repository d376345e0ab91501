// Axis stencils on few real points (point.hip).
#pragma once

#include "stencil.h"

namespace gfd {

// Most points (all grids) for one point per thread.  Full rows against this,
// us, FP64 Laplacians with inputs in rotation (and repeated on one): R = 1 5 x
// 48^3 5.8 / 5.4 (5.5 / 4.8), 7 x 48^3 6.2 / 6.4 (5.8 / 5.8); R = 2 4 x 150x32x26
// 6.1 / 5.6 (5.9 / 5.9), 5 x 48^3 6.7 / 6.8 (5.9 / 6.4); R = 3 5 x 48^3 9.3 / 8.7
// (8.4 / 7.9); R = 4 80^3 10.1 / 9.0 (9.3 / 8.7), 5 x 48^3 10.2 / 10.1 (9.4 / 9.4).
// A single axis (2R + 1 loads): along x at R = 4, the nearest, 6 x 48^3 0.93
// and 7 x 48^3 0.98 of the rows' time, along y and z 0.70 to 0.96 up to 1.3
// million points.  Against the march on grids the rows do not take: 5 x 47^3
// R = 2 6.5 / 5.9, R = 4 9.6 / 8.7; 6 x 47^3 6.9 / 6.8, 10.0 / 10.3.  FP32:
// whole solves with R = 3 sweeps, 96^3 2.58 / 2.28 ms, 128^3 3.00 / 3.33 ms.
constexpr double PT_MAX64[MAXR_FAST] = {650e3, 500e3, 600e3, 540e3};
constexpr double PT_MAX64_LINE = 750e3, PT_MAX64_ODD = 600e3;
constexpr double PT_MAX32 = 1000e3;

bool point_fits(const AxisStencil& st, int dtype, const int n[3], long nin,
                int epi);
int launch_point(const AxisStencil& st, int dtype, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out);

}  // namespace gfd
