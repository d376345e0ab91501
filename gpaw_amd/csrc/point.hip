// Axis stencils on few real points: one point per thread, every neighbour
// loaded directly.
//
// The marching kernels read each value once, but a block walks through its
// planes one latency after another; on arrays that the caches hold and that
// fill the chip only a few times over, one load latency for everything is
// faster (limits in point.h).  k_point issues its 6R + 1 loads at once, with the
// wrapped offsets from compares and selects, and has the accumulation order
// (z, y, x) and the epilogues of the full-row kernel.
#include "point.h"

#include <algorithm>

#include "stencil_dev.h"

namespace gfd {

constexpr int PT_NT = 256;

template <typename T>
struct PtArgs {
    const T* in;
    void* out;
    const void* aux;
    int n0, n1, n2;
    unsigned ng, total;
    int per0, per1, per2;
    int nblocks;
    double c0, w, s;
    int negate;
    int has0, has1, has2;
    double cp[3][MAXR_FAST], cm[3][MAXR_FAST];
    double* partial;
    const double* pot;
    const double* shift;
};

template <typename T, int R, int EPI>
__global__ void __launch_bounds__(PT_NT) k_point(PtArgs<T> a)
{
    const int L = xcd_remap(blockIdx.x, a.nblocks);
    const unsigned id = (unsigned)L * PT_NT + threadIdx.x;
    double nrm = 0.0;
    if (id < a.total) {
        const unsigned b = id / a.ng;
        const unsigned p = id - b * a.ng;
        const unsigned q = p / (unsigned)a.n2;
        const int i2 = (int)(p - q * a.n2);
        const int i0 = (int)(q / (unsigned)a.n1);
        const int i1 = (int)(q - (unsigned)i0 * a.n1);
        const T* g = a.in + (size_t)b * a.ng;
        const int plane = a.n1 * a.n2;
        const T v = g[p];
        T acc = zero_of<T>();
        // both neighbours at distance k along an axis of stride st
        auto axis = [&](int has, int i, int n, int per, int st,
                        const double* cp, const double* cm) {
            if (!has) return;
            T up[R], dn[R];
#pragma unroll
            for (int k = 1; k <= R; k++) {
                const int hi = i + k >= n ? i + k - n : i + k;
                const int lo = i < k ? i - k + n : i - k;
                const bool oh = per || i + k < n, ol = per || i >= k;
                const T h = g[(int)p + (oh ? hi - i : 0) * st];
                const T l = g[(int)p + (ol ? lo - i : 0) * st];
                up[k - 1] = oh ? h : zero_of<T>();
                dn[k - 1] = ol ? l : zero_of<T>();
            }
#pragma unroll
            for (int k = 0; k < R; k++) {
                acc = fmac(acc, (T)cp[k], up[k]);
                acc = fmac(acc, (T)cm[k], dn[k]);
            }
        };
        axis(a.has2, i2, a.n2, a.per2, 1, a.cp[2], a.cm[2]);
        axis(a.has1, i1, a.n1, a.per1, a.n2, a.cp[1], a.cm[1]);
        axis(a.has0, i0, a.n0, a.per0, plane, a.cp[0], a.cm[0]);
        if constexpr (EPI == EPI_POT) {
            T r = fmac(fmac(acc, a.c0, v), a.pot[p], v);
            if (a.shift) r = fmac(r, -a.shift[b], v);
            ((T*)a.out)[id] = r;
        } else if constexpr (EPI == EPI_RESN) {
            ((float*)a.out)[id] = (float)epi_apply<T, EPI_RESID>(
                acc, v, ((const T*)a.aux)[id], a.c0, a.w, a.s, a.negate,
                nrm);
        } else if constexpr (EPI == EPI_UPDW) {
            const T av = to_narrow(((const double*)a.aux)[id]);
            ((double*)a.out)[id] = to_wide(epi_apply<T, EPI_UPDATE>(
                acc, v, av, a.c0, a.w, a.s, a.negate, nrm));
        } else {
            T av = zero_of<T>();
            if constexpr (EPI != EPI_PLAIN) av = ((const T*)a.aux)[id];
            ((T*)a.out)[id] = epi_apply<T, EPI>(acc, v, av, a.c0, a.w, a.s,
                                                a.negate, nrm);
        }
    }
    if ((EPI == EPI_RESID || EPI == EPI_RESN) && a.partial)
        block_sum_store(nrm, a.partial, L);
}

template <typename T, int R, int EPI>
static int pt_launch(const AxisStencil& st, const int n[3], const BC& bc,
                     const void* in, void* out, long nin, const EpiArgs& ea,
                     hipStream_t s, int* nbo)
{
    PtArgs<T> a;
    a.in = (const T*)in;
    a.out = out;
    a.aux = ea.aux;
    a.n0 = n[0];
    a.n1 = n[1];
    a.n2 = n[2];
    a.ng = (unsigned)((long)n[0] * n[1] * n[2]);
    a.total = (unsigned)(a.ng * nin);
    a.per0 = bc.periodic[0];
    a.per1 = bc.periodic[1];
    a.per2 = bc.periodic[2];
    a.nblocks = (int)((a.total + PT_NT - 1) / PT_NT);
    a.c0 = ea.c0;
    a.w = ea.w;
    a.s = ea.s;
    a.negate = ea.negate;
    a.has0 = st.has[0];
    a.has1 = st.has[1];
    a.has2 = st.has[2];
    for (int c = 0; c < 3; c++)
        for (int k = 0; k < MAXR_FAST; k++) {
            a.cp[c][k] = st.cp[c][k];
            a.cm[c][k] = st.cm[c][k];
        }
    a.partial = ea.partial;
    a.pot = ea.pot;
    a.shift = ea.shift;
    (void)hipGetLastError();
    hipLaunchKernelGGL((k_point<T, R, EPI>), dim3((unsigned)a.nblocks),
                       dim3(PT_NT), 0, s, a);
    GFD_LAUNCH_CHECK();
    if (nbo) *nbo = a.nblocks;
    return OK;
}

template <typename T, int EPI>
static int pt_radius(const AxisStencil& st, const int n[3], const BC& bc,
                     const void* in, void* out, long nin, const EpiArgs& ea,
                     hipStream_t s, int* nbo)
{
    switch (st.R) {
    case 1: return pt_launch<T, 1, EPI>(st, n, bc, in, out, nin, ea, s, nbo);
    case 2: return pt_launch<T, 2, EPI>(st, n, bc, in, out, nin, ea, s, nbo);
    case 3: return pt_launch<T, 3, EPI>(st, n, bc, in, out, nin, ea, s, nbo);
    case 4: return pt_launch<T, 4, EPI>(st, n, bc, in, out, nin, ea, s, nbo);
    }
    set_error("point stencil: radius %d", st.R);
    return ENOTSUP_;
}

bool point_fits(const AxisStencil& st, int dtype, const int n[3], long nin,
                int epi)
{
    const bool has = (dtype == 0 && epi != EPI_UPDW) ||
                     (dtype == 2 && epi != EPI_POT && epi != EPI_RESN);
    if (!has || st.R < 1 || st.R > MAXR_FAST || n[0] < st.R ||
        n[1] < st.R || n[2] < st.R)
        return false;
    const bool line = (st.has[0] != 0) + (st.has[1] != 0) +
                          (st.has[2] != 0) == 1;
    double most = dtype == 2 ? PT_MAX32
                  : line     ? PT_MAX64_LINE
                             : PT_MAX64[st.R - 1];
    if (!row_stencil_fits(st, dtype, n, nin))
        most = std::max(most, PT_MAX64_ODD);
    return (double)n[0] * n[1] * n[2] * (double)nin <= most;
}

int launch_point(const AxisStencil& st, int dtype, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out)
{
#define GFD_PT(T, EPI)                                                      \
    case EPI:                                                               \
        return pt_radius<T, EPI>(st, n, bc, in, out, nin, ea, s, nblocks_out)
    if (dtype == 0) {
        switch (epi) {
            GFD_PT(double, EPI_PLAIN);
            GFD_PT(double, EPI_RELAX);
            GFD_PT(double, EPI_RESID);
            GFD_PT(double, EPI_UPDATE);
            GFD_PT(double, EPI_POT);
            GFD_PT(double, EPI_RESN);
        }
    } else if (dtype == 2) {
        switch (epi) {
            GFD_PT(float, EPI_PLAIN);
            GFD_PT(float, EPI_RELAX);
            GFD_PT(float, EPI_RESID);
            GFD_PT(float, EPI_UPDATE);
            GFD_PT(float, EPI_UPDW);
        }
    }
#undef GFD_PT
    set_error("point stencil: data type %d / epilogue %d not built", dtype,
              epi);
    return ENOTSUP_;
}

}  // namespace gfd
