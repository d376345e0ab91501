// Stencil kernels for gfx950.
//
// k_general computes `out = sum_p c_p in(x + o_p)` over batches of grids for
// any offsets, with the halo taken by index wrap (no padded copies): one
// output point per thread with direct, cache-served neighbour loads.  It
// takes what the full-row kernel (rows_kernel.h) and the direction march
// (dirmarch_kernel.h) do not: points off every straight line through the
// centre, more or longer lines than those hold, duplicate points.
//
// It finishes with one of the epilogues of stencil.h, which fuse the Jacobi
// update, the residual (+ its squared norm) and the preconditioner's
// residual-update into the same pass.
#include "stencil.h"
#include "stencil_dev.h"

#include <algorithm>
#include <cstdarg>
#include <mutex>

namespace gfd {

// ------------------------------------------------------------ general

template <typename T>
struct GenArgs {
    const T* in;
    T* out;
    const T* aux;
    int n0, n1, n2;
    long ng, total;
    int P, centre;
    const double* coef;
    const int* off;
    double c0, w, s;
    int negate;
    BC bc;
    double* partial;
    const double* pot;
    const double* shift;
};

constexpr int GEN_BLOCK = 256;

template <typename T, int EPI>
__global__ void __launch_bounds__(GEN_BLOCK) k_general(GenArgs<T> a)
{
    typedef typename ScalarOf<T>::type S;
    const long gid = (long)blockIdx.x * GEN_BLOCK + threadIdx.x;
    double nrm = 0.0;
    if (gid < a.total) {
        long b;
        int i0, i1, i2;
        flat_split(gid, a.total, a.ng, a.n1, a.n2, b, i0, i1, i2);
        const T* __restrict__ g = a.in + b * a.ng;
        T acc = zero_of<T>();
        for (int c = 0; c < a.P; c++) {
            if (c == a.centre) continue;
            int j0 = i0 + a.off[3 * c], j1 = i1 + a.off[3 * c + 1],
                j2 = i2 + a.off[3 * c + 2];
            double2 f = make_double2(1.0, 0.0);
            bool ph = false;
            bool ok = wrap_full(j0, a.n0, a.bc.periodic[0], a.bc.phase[0][0],
                                a.bc.phase[0][1], f, ph);
            ok = ok && wrap_full(j1, a.n1, a.bc.periodic[1],
                                 a.bc.phase[1][0], a.bc.phase[1][1], f, ph);
            ok = ok && wrap_full(j2, a.n2, a.bc.periodic[2],
                                 a.bc.phase[2][0], a.bc.phase[2][1], f, ph);
            if (!ok) continue;
            T v = g[((long)j0 * a.n1 + j1) * a.n2 + j2];
            v = scale_by<T>(v, f, ph);
            acc = fmac(acc, (S)a.coef[c], v);
        }
        const T v = g[((long)i0 * a.n1 + i1) * a.n2 + i2];
        if constexpr (EPI == EPI_POT) {
            typedef typename ScalarOf<T>::type S;
            T r = fmac(fmac(acc, (S)a.c0, v), (S)a.pot[gid - b * a.ng], v);
            if (a.shift) r = fmac(r, -(S)a.shift[b], v);
            a.out[gid] = r;
        } else if constexpr (EPI == EPI_RESN) {
            ((float*)(void*)a.out)[gid] = (float)epilogue<T, EPI_RESID>(
                acc, v, a.aux, gid, a.c0, a.w, a.s, a.negate, nrm);
        } else if constexpr (EPI == EPI_UPDW) {
            typedef typename WideOf<T>::type WT;
            const T av = to_narrow(((const WT*)(const void*)a.aux)[gid]);
            const T r = epi_apply<T, EPI_UPDATE>(acc, v, av, a.c0, a.w, a.s,
                                                 a.negate, nrm);
            ((WT*)(void*)a.out)[gid] = to_wide(r);
        } else {
            a.out[gid] = epilogue<T, EPI>(acc, v, a.aux, gid, a.c0, a.w, a.s,
                                          a.negate, nrm);
        }
    }
    if ((EPI == EPI_RESID || EPI == EPI_RESN) && a.partial)
        block_sum_store(nrm, a.partial, blockIdx.x);
}

// ------------------------------------------------------------ reduction

__global__ void __launch_bounds__(1024)
k_sum_partials(const double* __restrict__ p, long np, double* out)
{
    double s = 0.0;
    for (long i = threadIdx.x; i < np; i += 1024) s += p[i];
    __shared__ double red[16];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < 16; i++) t += red[i];
        *out = t;
    }
}

int launch_sum_partials(const double* partial, long np, double* result,
                        hipStream_t stream)
{
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, stream,
                       partial, np, result);
    GFD_LAUNCH_CHECK();
    return OK;
}

// ------------------------------------------------------------ host side

long general_stencil_max_blocks(const int n[3], long nin)
{
    return ((long)n[0] * n[1] * n[2] * nin + GEN_BLOCK - 1) / GEN_BLOCK;
}

template <typename T, int EPI>
static int launch_gen_t(const GeneralStencil& st, const int n[3],
                        const BC& bc, const void* in, void* out, long nin,
                        const EpiArgs& ea, hipStream_t stream, int* nbo)
{
    GenArgs<T> a;
    a.in = (const T*)in;
    a.out = (T*)out;
    a.aux = (const T*)ea.aux;
    a.n0 = n[0];
    a.n1 = n[1];
    a.n2 = n[2];
    a.ng = (long)n[0] * n[1] * n[2];
    a.total = a.ng * nin;
    a.P = st.P;
    a.centre = st.centre;
    a.coef = st.coef;
    a.off = st.off;
    a.c0 = ea.c0;
    a.w = ea.w;
    a.s = ea.s;
    a.negate = ea.negate;
    a.bc = bc;
    a.partial = ea.partial;
    a.pot = ea.pot;
    a.shift = ea.shift;
    const long nb = (a.total + GEN_BLOCK - 1) / GEN_BLOCK;
    if (nb <= 0) return OK;
    if (nb > 0x7fffffffL) {
        set_error("too many blocks (%ld)", nb);
        return ENOTSUP_;
    }
    hipLaunchKernelGGL((k_general<T, EPI>), dim3((unsigned)nb),
                       dim3(GEN_BLOCK), 0, stream, a);
    GFD_LAUNCH_CHECK();
    if (nbo) *nbo = (int)nb;
    return OK;
}

int launch_general_stencil(const GeneralStencil& st, int dtype,
                           const int n[3], const BC& bc, const void* in,
                           void* out, long nin, int epi, const EpiArgs& ea,
                           hipStream_t stream, int* nblocks_out)
{
    if (dtype == 0) {
        switch (epi) {
        case EPI_PLAIN: return launch_gen_t<double, EPI_PLAIN>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RELAX: return launch_gen_t<double, EPI_RELAX>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RESID: return launch_gen_t<double, EPI_RESID>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_UPDATE: return launch_gen_t<double, EPI_UPDATE>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_POT: return launch_gen_t<double, EPI_POT>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RESN: return launch_gen_t<double, EPI_RESN>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        }
    } else if (dtype == 1) {
        switch (epi) {
        case EPI_POT: return launch_gen_t<double2, EPI_POT>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_PLAIN: return launch_gen_t<double2, EPI_PLAIN>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RESID: return launch_gen_t<double2, EPI_RESID>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_UPDATE: return launch_gen_t<double2, EPI_UPDATE>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        }
    } else if (dtype == 2) {
        switch (epi) {
        case EPI_PLAIN: return launch_gen_t<float, EPI_PLAIN>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RELAX: return launch_gen_t<float, EPI_RELAX>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RESID: return launch_gen_t<float, EPI_RESID>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_UPDATE: return launch_gen_t<float, EPI_UPDATE>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_UPDW: return launch_gen_t<float, EPI_UPDW>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        }
    } else if (dtype == 3) {
        switch (epi) {
        case EPI_PLAIN: return launch_gen_t<float2, EPI_PLAIN>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_RESID: return launch_gen_t<float2, EPI_RESID>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_UPDATE: return launch_gen_t<float2, EPI_UPDATE>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        case EPI_UPDW: return launch_gen_t<float2, EPI_UPDW>(st, n, bc, in, out, nin, ea, stream, nblocks_out);
        }
    }
    set_error("general stencil: unsupported dtype %d / epilogue %d", dtype,
              epi);
    return ENOTSUP_;
}

}  // namespace gfd
