#include "dirmarch_kernel.h"

namespace gfd {

int dirmarch_f64(const DirStencil& d, const DirTile& t, const int n[3],
                 const BC& bc, const void* in, void* out, long nin, int epi,
                 const EpiArgs& ea, hipStream_t s, int* nblocks_out)
{
    return dm_launch<double>(d, t, n, bc, in, out, nin, epi, ea, s, nblocks_out);
}

}  // namespace gfd
