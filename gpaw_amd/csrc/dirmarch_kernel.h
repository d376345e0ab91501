// k_dirmarch: one pass of a direction stencil (dirmarch.h).  Included by the
// dirmarch_*.hip units, one per data type.
//
// A block owns a (ty x tz) tile of one grid and marches along x.  Each input
// plane of the tile with its R-wide halo is staged in LDS (double buffered,
// one barrier per plane; every thread loads its share of the extended tile,
// so halo and own points are one stream of loads) and used once for
// everything it contributes to: a thread keeps one accumulator per output
// plane x - R .. x + R of its column, adds the in-plane directions to the
// middle one and every k-th point of a direction (1, dy, dz) to the one k
// planes away, and stores the oldest.  The plane loop is unrolled by the
// 2R + 1 accumulators, which are thereby renamed instead of moved.
//
// The centre value waits in a queue of R + 1 for its output plane and is
// added last: the largest term of the sum, whose rounding every term after
// it would inherit.
//
// All global traffic goes through per-plane buffer resources: zero
// boundaries and idle lanes are out-of-range offsets, not branches.
//
// What bounds it, by counters: HBM traffic, of which halo rows read again are
// a third or more (48 c128 grids of 128^3, H psi - eps psi: 703 us, 2.4 GiB
// fetched for 1.5, 5.9 TB/s in all; k_xrow 1006 us at 2 waves per SIMD; 40 f64
// grids of 87x103x95, H psi: 174 us, 573 MiB fetched for 268, 5.1 TB/s; one
// point per thread with every index wrapped took 790 us); for the skew
// stencils the LDS reads (18 of 16 bytes beside the own point per complex
// point of the 25-point hexagonal Laplacian, the LDS unit active 70 % of the
// time and a third of that on bank conflicts: 24 grids of 60x60x84 64 us, 60
// repeated on one input; wrapped point by point 247 us).
#pragma once

#include "dirmarch.h"

#include "batch.h"
#include "rows.h"
#include "stencil_dev.h"

namespace gfd {

constexpr int DM_NT = 512;  // most threads of a block

template <typename T>
struct DmArgs {
    const T* in;
    void* out;
    const void* aux;
    int n0, n1, n2;
    int tz, ty, tiles_z, tiles_y, chunks_x, xchunk, nblocks;
    int epi;
    double c0, w, s;
    int negate;
    DirStencil st;
    BC bc;
    double* partial;
    const double* shift;
};

template <typename T>
__device__ inline void dm_store(T v, __amdgpu_buffer_rsrc_t r, unsigned off)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(T) <= 8)
        bstore(v, r, off);
    else
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r,
                                               (int)off, 0, 0);
}

__device__ inline float dm_narrow(double v) { return (float)v; }
__device__ inline float2 dm_narrow(double2 v)
{
    return make_float2((float)v.x, (float)v.y);
}

// what an epilogue reads beside the stencil input
enum DmAux : int { DM_NONE = 0, DM_SAME = 1, DM_POT = 2, DM_WIDE = 3 };

// AUX: DmAux.  HM: staged elements per thread.  NARROW: FP64 input, result
// stored as FP32 (EPI_RESN).
// FORM:
//   DM_FULL: every direction of the form is there with equal coefficients on
//     both sides of the centre (a Laplacian).  Then nothing is tested in the
//     plane loop, whose many scalar tests and branches were what bound the
//     first version (142 scalar instructions, 20 of them branches, beside 38
//     vector ones per plane), and one copy of the coefficients stays in
//     scalar registers.
//   DM_LINE + axis: that axis line alone (a gradient).  Along x nothing is
//     staged: a thread's own column is all it reads.  Along y or z a plane
//     stands by itself, with a halo on that axis only.
//   DM_GENERAL: any set of directions, each tested per plane.
enum DmForm : int { DM_GENERAL = 0, DM_FULL = 1, DM_LINE = 2 };

template <typename T, int R, int NI, int NM, int AUX, int HM, int FORM,
          bool NARROW>
__global__ void __launch_bounds__(DM_NT) k_dirmarch(DmArgs<T> a)
{
    typedef typename ScalarOf<T>::type S;
    typedef typename WideOf<T>::type WT;
    typedef typename std::conditional<
        AUX == DM_POT, double,
        typename std::conditional<AUX == DM_WIDE, WT, T>::type>::type TA;
    typedef typename std::conditional<
        NARROW, float,
        typename std::conditional<AUX == DM_WIDE, WT, T>::type>::type TO;
    constexpr bool FULL = FORM == DM_FULL;
    constexpr int LINE = FORM < DM_LINE ? -1 : FORM - DM_LINE;
    constexpr DirHalo H = dir_halo(R, LINE);
    constexpr int U = 2 * H.x + 1;
    constexpr bool CPLX = IsCplx<T>::value;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* lds = reinterpret_cast<T*>(smem_raw);

    const int L = xcd_remap(blockIdx.x, a.nblocks);
    int rem = L;
    const int zt = rem % a.tiles_z;
    rem /= a.tiles_z;
    const int yt = rem % a.tiles_y;
    rem /= a.tiles_y;
    const int cx = rem % a.chunks_x;
    const long b = rem / a.chunks_x;

    const int tid = threadIdx.x, NT = blockDim.x;
    const int n0 = a.n0, n1 = a.n1, n2 = a.n2;
    const long ng = (long)n1 * n2 * n0;
    const unsigned plane = (unsigned)n1 * (unsigned)n2;
    const int z0 = zt * a.tz, y0 = yt * a.ty;
    const int xs = cx * a.xchunk, xe = min(xs + a.xchunk, n0);
    const int LW = a.tz + 2 * H.z, LSZ = (a.ty + 2 * H.y) * LW;
    const int buf1 = HM * NT;  // elements of one buffer (LSZ at most)
    const BC& bc = a.bc;

    // staged elements tid + m NT of the extended tile: offset in the plane
    // (BXM_OOB: zero or unused) and Bloch factor of the y and z wraps
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
            int y = y0 + row - H.y, z = z0 + (e - row * LW) - H.z;
            // beyond the halo of the last row or column: never read
            if (y < n1 + H.y && z < n2 + H.z &&
                wrap_full(z, n2, bc.periodic[2], bc.phase[2][0],
                          bc.phase[2][1], hf[m], hph[m]) &&
                wrap_full(y, n1, bc.periodic[1], bc.phase[1][0],
                          bc.phase[1][1], hf[m], hph[m]))
                hoff[m] = (unsigned)(y * n2 + z) * (unsigned)sizeof(T);
        }
    }
    // own point
    const int tr = tid / a.tz, tc = tid - tr * a.tz;
    const bool on = tr < a.ty && y0 + tr < n1 && z0 + tc < n2;
    const int lown = (min(tr, a.ty - 1) + H.y) * LW + tc + H.z;
    const unsigned oidx = (unsigned)((y0 + tr) * n2 + z0 + tc);
    const unsigned ooff = on ? oidx * (unsigned)sizeof(TO) : BXM_OOB;
    const unsigned aoff = on ? oidx * (unsigned)sizeof(TA) : BXM_OOB;

    // resource of plane x of an array of E (empty unless ok)
    auto plane_at = [&](const void* base, int x, unsigned es, bool ok) {
        const unsigned pb = plane * es;
        return brsrc((const char*)base + (unsigned long)pb * (unsigned)x,
                     ok ? pb : 0u);
    };
    const void* gin = a.in + b * ng;
    const void* gaux = (const TA*)a.aux + (AUX == DM_POT ? 0 : b * ng);
    void* gout = (TO*)a.out + b * ng;
    T hv[HM];
    double2 fx = make_double2(1.0, 0.0);
    bool phx = false;
    // input plane x in [-R, n0 + R): wrapped at most once (n0 >= R), empty
    // beyond a zero boundary
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
    TA av{};
    // auxiliary operand of output plane x (the chunk's nearest plane before
    // and after it: the array has no others)
    auto ld_aux = [&](int x) {
        if constexpr (AUX != DM_NONE)
            av = bload<TA>(plane_at(gaux, min(max(x, xs), xe - 1),
                                    sizeof(TA), true),
                           aoff);
    };
    auto cm = [](const DirLine& l, int k) {
        return (S)(FULL ? l.p[k - 1] : l.m[k - 1]);
    };
    // the point k steps along l is there (k < 0: behind)
    auto has = [](const DirLine& l, int k) {
        return (l.has >> (k > 0 ? k - 1 : MAXR_FAST - k - 1) & 1u) != 0;
    };
    S shift = (S)0;
    if constexpr (AUX == DM_POT)
        if (a.shift) shift = -(S)a.shift[b];

    T acc[U];
#pragma unroll
    for (int j = 0; j < U; j++) acc[j] = zero_of<T>();
    T vq[H.x + 1];  // centre values of planes x - H.x .. x
#pragma unroll
    for (int j = 0; j <= H.x; j++) vq[j] = zero_of<T>();
    double nrm = 0.0;

    ld_plane(xs - H.x);
    ld_aux(xs);
    int cur = 0;
    for (int xb = xs - H.x; xb < xe + H.x; xb += U) {
        cfor<U>([&](auto uc) {
            constexpr int u = uc;
            const int x = xb + u;
            if (x >= xe + H.x) return;
            T* buf = lds + cur;
            cur = buf1 - cur;
            T v;
#pragma unroll
            for (int m = 0; m < HM; m++) {
                v = hv[m];
                if constexpr (CPLX) {
                    if (hph[m]) v = scale_by<T>(v, hf[m], true);
                    if (phx) v = scale_by<T>(v, fx, true);
                }
                if constexpr (LINE != 0) buf[tid + m * NT] = v;
            }
            ld_plane(min(x + 1, xe + H.x - 1));
            if constexpr (LINE != 0) __syncthreads();

            // accumulator of output plane x + j: (u + H.x + j) mod U
            auto at = [&](auto j) -> T& {
                constexpr int i = (u + H.x + decltype(j)::value + U) % U;
                return acc[i];
            };
            constexpr std::integral_constant<int, 0> here;
            constexpr std::integral_constant<int, -H.x> oldest;
            const T* p = buf + lown;
            // (along x the one staged point is the thread's own)
            if constexpr (LINE != 0) v = p[0];
            cfor<H.x>([&](auto j) { vq[j] = vq[j + 1]; });
            vq[H.x] = v;
            T mid = at(here);
            // in-plane direction l with its points o elements apart
            auto inplane = [&](const DirLine& l, int o) {
                if (FORM != DM_GENERAL || l.on == DIR_ALL) {
#pragma unroll
                    for (int k = 1; k <= R; k++) {
                        mid = fmac(mid, (S)l.p[k - 1], p[k * o]);
                        mid = fmac(mid, cm(l, k), p[-k * o]);
                    }
                } else if (l.on != DIR_NONE) {
#pragma unroll
                    for (int k = 1; k <= R; k++) {
                        if (has(l, k)) mid = fmac(mid, (S)l.p[k - 1], p[k * o]);
                        if (has(l, -k)) mid = fmac(mid, cm(l, k), p[-k * o]);
                    }
                }
            };
            if constexpr (LINE < 0 || LINE == 2) inplane(a.st.in[0], 1);
            if constexpr (LINE < 0 || LINE == 1) inplane(a.st.in[1], LW);
#pragma unroll
            for (int i = 2; i < NI; i++)
                inplane(a.st.in[i], a.st.in[i].dy * LW + a.st.in[i].dz);
            at(here) = mid;
            // direction l off the x axis: the point k steps ahead of output
            // x - k, behind output x + k
            auto across = [&](const DirLine& l, auto&& point) {
                auto step = [&](auto all, auto k0) {
                    constexpr int k = k0 + 1;
                    std::integral_constant<int, -k> ahead;
                    std::integral_constant<int, k> behind;
                    if (all || has(l, k))
                        at(ahead) = fmac(at(ahead), (S)l.p[k - 1], point(k));
                    if (all || has(l, -k))
                        at(behind) = fmac(at(behind), cm(l, k), point(-k));
                };
                if (FORM != DM_GENERAL || l.on == DIR_ALL)
                    cfor<R>([&](auto k) { step(std::true_type{}, k); });
                else if (l.on != DIR_NONE)
                    cfor<R>([&](auto k) { step(std::false_type{}, k); });
            };
            if constexpr (LINE < 1) across(a.st.x, [&](int) { return v; });
#pragma unroll
            for (int i = 0; i < NM; i++) {
                const int o = a.st.mix[i].dy * LW + a.st.mix[i].dz;
                across(a.st.mix[i], [&](int k) { return p[k * o]; });
            }
            // output plane x - H.x is complete (before the chunk: not stored)
            const int xo = x - H.x;
            T r = at(oldest);
            const T vo = vq[0];
            if constexpr (AUX == DM_POT) {
                r = fmac(fmac(r, (S)a.c0, vo), (S)av, vo);
                if (a.shift) r = fmac(r, shift, vo);
            } else if constexpr (AUX == DM_NONE) {
                r = fmac(r, (S)a.c0, vo);
            } else {
                T ax;
                if constexpr (AUX == DM_WIDE) ax = dm_narrow(av);
                else ax = av;
                if (a.epi == EPI_RELAX)
                    r = epi_apply<T, EPI_RELAX>(r, vo, ax, a.c0, a.w, a.s,
                                                a.negate, nrm);
                else if (a.epi == EPI_RESID) {
                    r = fmac(r, (S)a.c0, vo) - ax;
                    if (on && xo >= xs) nrm += sq(r);
                } else
                    r = epi_apply<T, EPI_UPDATE>(r, vo, ax, a.c0, a.w, a.s,
                                                 a.negate, nrm);
            }
            TO ro;
            if constexpr (NARROW) ro = (float)r;
            else if constexpr (AUX == DM_WIDE) ro = to_wide(r);
            else ro = r;
            dm_store(ro, plane_at(gout, xo, sizeof(TO), xo >= xs), ooff);
            at(oldest) = zero_of<T>();
            // reloaded once used: a copy of a value in flight would wait
            ld_aux(xo + 1);
        });
    }
    if constexpr (AUX == DM_SAME)
        if (a.partial) block_sum_store(nrm, a.partial, L);
}

template <typename T, int R, int NI, int NM, int AUX, int HM, int FORM,
          bool NARROW>
static int dm_launch_t(const DirStencil& d, const DirTile& t, const int n[3],
                       const BC& bc, const void* in, void* out, long nin,
                       int epi, const EpiArgs& ea, hipStream_t s, int* nbo)
{
    DmArgs<T> a;
    a.in = (const T*)in;
    a.out = out;
    a.aux = AUX == DM_POT ? (const void*)ea.pot : ea.aux;
    a.n0 = n[0];
    a.n1 = n[1];
    a.n2 = n[2];
    a.tz = t.tz;
    a.ty = t.ty;
    a.tiles_z = ceil_div(n[2], t.tz);
    a.tiles_y = ceil_div(n[1], t.ty);
    a.xchunk = t.xchunk;
    a.chunks_x = ceil_div(n[0], t.xchunk);
    const long nb = (long)a.tiles_z * a.tiles_y * a.chunks_x * nin;
    const int threads = t.threads;
    constexpr DirHalo H = dir_halo(R, FORM < DM_LINE ? -1 : FORM - DM_LINE);
    const long lsz = (long)(t.tz + 2 * H.z) * (t.ty + 2 * H.y);
    if (nb <= 0) return OK;
    if (nb > 0x7fffffffL || threads > DM_NT || threads < t.tz * t.ty ||
        lsz > (long)HM * threads) {
        set_error("direction march: %ld blocks of %d x %d do not fit", nb,
                  t.ty, t.tz);
        return ENOTSUP_;
    }
    a.nblocks = (int)nb;
    a.epi = epi == EPI_RESN ? (int)EPI_RESID : epi;
    a.c0 = ea.c0;
    a.w = ea.w;
    a.s = ea.s;
    a.negate = ea.negate;
    a.st = d;
    a.bc = bc;
    a.partial = epi == EPI_RESID || epi == EPI_RESN ? ea.partial : nullptr;
    a.shift = ea.shift;
    (void)hipGetLastError();
    hipLaunchKernelGGL((k_dirmarch<T, R, NI, NM, AUX, HM, FORM, NARROW>),
                       dim3((unsigned)nb), dim3(threads),
                       FORM == DM_LINE
                           ? 0
                           : 2 * (size_t)HM * threads * sizeof(T),
                       s, a);
    GFD_LAUNCH_CHECK();
    if (nbo) *nbo = (int)nb;
    return OK;
}

template <typename T, int R, int NI, int NM, int AUX, int FORM, bool NARROW>
static int dm_launch_h(const DirStencil& d, const DirTile& t, const int n[3],
                       const BC& bc, const void* in, void* out, long nin,
                       int epi, const EpiArgs& ea, hipStream_t s, int* nbo)
{
#define GFD_DM(HM)                                                          \
    return dm_launch_t<T, R, NI, NM, AUX, HM, FORM, NARROW>(                \
        d, t, n, bc, in, out, nin, epi, ea, s, nbo)
    constexpr DirHalo H = dir_halo(R, FORM < DM_LINE ? -1 : FORM - DM_LINE);
    const long lsz = (long)(t.tz + 2 * H.z) * (t.ty + 2 * H.y);
    if constexpr (FORM == DM_LINE) GFD_DM(1);
    else {
        if constexpr (FORM != DM_GENERAL || (NM == 0 && R <= DM_RSKEW))
            if (lsz <= 2L * t.threads) GFD_DM(2);
        GFD_DM(4);
    }
#undef GFD_DM
}

template <typename T, int R, int NI, int NM, int FORM>
static int dm_launch_e(const DirStencil& d, const DirTile& t, const int n[3],
                       const BC& bc, const void* in, void* out, long nin,
                       int epi, const EpiArgs& ea, hipStream_t s, int* nbo)
{
#define GFD_DM(AUX, NARROW)                                                 \
    return dm_launch_h<T, R, NI, NM, AUX, FORM, NARROW>(                    \
        d, t, n, bc, in, out, nin, epi, ea, s, nbo)
    if constexpr (FORM >= DM_LINE) GFD_DM(DM_NONE, false);  // EPI_PLAIN
    else
    switch (epi) {
    case EPI_PLAIN: GFD_DM(DM_NONE, false);
    case EPI_RELAX:
    case EPI_RESID:
    case EPI_UPDATE: GFD_DM(DM_SAME, false);
    case EPI_POT:
        if constexpr (sizeof(typename ScalarOf<T>::type) == 8)
            GFD_DM(DM_POT, false);
        break;
    case EPI_UPDW:
        if constexpr (sizeof(typename ScalarOf<T>::type) == 4)
            GFD_DM(DM_WIDE, false);
        break;
    case EPI_RESN:
        if constexpr (std::is_same<T, double>::value) GFD_DM(DM_SAME, true);
        break;
    }
#undef GFD_DM
    set_error("direction march: epilogue %d not built", epi);
    return ENOTSUP_;
}

template <typename T, int R>
static int dm_launch_r(const DirStencil& d, const DirTile& t, const int n[3],
                       const BC& bc, const void* in, void* out, long nin,
                       int epi, const EpiArgs& ea, hipStream_t s, int* nbo)
{
#define GFD_DM(NI, NM, FORM)                                                \
    return dm_launch_e<T, R, NI, NM, FORM>(d, t, n, bc, in, out, nin, epi,  \
                                           ea, s, nbo)
    constexpr bool WIDE = sizeof(typename ScalarOf<T>::type) == 8;
    if constexpr (WIDE) {
        switch (dir_line(d, IsCplx<T>::value, epi)) {
        case 0: GFD_DM(2, 0, DM_LINE);
        case 1: GFD_DM(2, 0, DM_LINE + 1);
        case 2: GFD_DM(2, 0, DM_LINE + 2);
        }
    }
    if (d.full) {
        if (d.ni == 2 && d.nm == 0) GFD_DM(2, 0, DM_FULL);
        if constexpr (R <= DM_RSKEW) {
            if (d.ni == 2 && d.nm == 1) GFD_DM(2, 1, DM_FULL);
            if (d.ni == 3 && d.nm == 0) GFD_DM(3, 0, DM_FULL);
            if (d.ni == 3 && d.nm == 2) GFD_DM(3, 2, DM_FULL);
        }
    }
    // anything else: the general form of the directions, of the axes for
    // plain FP64 passes that need no more
    if constexpr (WIDE && R <= DM_RSKEW)
        if (d.ni == 2 && d.nm == 0 && epi == EPI_PLAIN)
            return dm_launch_h<T, R, 2, 0, DM_NONE, DM_GENERAL, false>(
                d, t, n, bc, in, out, nin, epi, ea, s, nbo);
    if constexpr (R <= DM_RSKEW) GFD_DM(3, 4, DM_GENERAL);
    else GFD_DM(2, 0, DM_GENERAL);
#undef GFD_DM
}

template <typename T>
static int dm_launch(const DirStencil& d, const DirTile& t, const int n[3],
                     const BC& bc, const void* in, void* out, long nin,
                     int epi, const EpiArgs& ea, hipStream_t s, int* nbo)
{
    switch (d.R) {
    case 1: return dm_launch_r<T, 1>(d, t, n, bc, in, out, nin, epi, ea, s, nbo);
    case 2: return dm_launch_r<T, 2>(d, t, n, bc, in, out, nin, epi, ea, s, nbo);
    case 3: return dm_launch_r<T, 3>(d, t, n, bc, in, out, nin, epi, ea, s, nbo);
    case 4: return dm_launch_r<T, 4>(d, t, n, bc, in, out, nin, epi, ea, s, nbo);
    }
    set_error("direction march: radius %d", d.R);
    return ENOTSUP_;
}

}  // namespace gfd
