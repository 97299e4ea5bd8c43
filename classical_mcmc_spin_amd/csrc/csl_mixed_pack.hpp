// csl_mixed_pack.hpp — packed partner tables of the mixed lattice's
// persistent and tangent kernels (host side, no HIP).
#pragma once

#include <cstddef>
#include <vector>

namespace cslh {

// Partner indices of every site of one species, 16 bits each, Z to a site:
// its cnt[p] partners (col[k * NP + p]), then unused slots, which the kernels
// gather too and multiply by a zero matrix.  An unused slot must therefore be
// a site whose value is as finite as the site's own field: the first partner,
// or for a site without any the same cell's site of the first sublattice.
// Both are cells of the lattice where p is one (what stage buffers in device
// memory hold for padding sites is never written), and padding (zero in LDS)
// where p is padding.
inline std::vector<unsigned short> packed_partners(const int* col, const int* cnt, int NP, int Z, int npad) {
    std::vector<unsigned short> q(size_t(NP) * Z);
    for (int p = 0; p < NP; ++p) {
        const int unused = cnt[p] > 0 ? col[p] : p % npad;
        for (int k = 0; k < Z; ++k)
            q[size_t(p) * Z + k] = static_cast<unsigned short>(k < cnt[p] ? col[size_t(k) * NP + p] : unused);
    }
    return q;
}

}  // namespace cslh
