// csl_mixed_pack.hpp — packed partner tables of the mixed lattice's
// persistent and tangent kernels (host side, no HIP).
#pragma once

#include <cstddef>
#include <vector>

namespace cslh {

// Partner indices of every site of one species, 16 bits each, Z to a site:
// its cnt[p] partners (col[k * NP + p]), then unused slots, which the kernels
// gather too and multiply by a zero matrix.  Zero times an infinity or a
// leftover of unwritten memory is not zero, so an unused slot repeats the
// site's first partner, and a site without partners (padding among them) has
// index npart, a record of zeros behind the partner species' npart records in
// LDS.
inline std::vector<unsigned short> packed_partners(const int* col, const int* cnt, int NP, int Z, int npart) {
    std::vector<unsigned short> q(size_t(NP) * Z);
    for (int p = 0; p < NP; ++p) {
        const int unused = cnt[p] > 0 ? col[p] : npart;
        for (int k = 0; k < Z; ++k)
            q[size_t(p) * Z + k] = static_cast<unsigned short>(k < cnt[p] ? col[size_t(k) * NP + p] : unused);
    }
    return q;
}

}  // namespace cslh
