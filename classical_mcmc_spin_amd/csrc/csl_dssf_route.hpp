// csl_dssf_route.hpp — which engine a structure-factor call takes and how
// many samples it transforms at a time (host side, no HIP).
#pragma once

#include <algorithm>
#include <cstddef>

namespace cslh {

struct DssfRoute {
    bool persistent;  // samples left by one launch (csl_dssf.hip), or the stage kernels sample by sample
    size_t nc;        // samples per transform
};

// `grid`: values of one sample (trajectories x sublattices x components x
// cells), `row`: those of S(q, t) (without the sublattices).  The samples may
// take a quarter of the memory available, all buffers three quarters: samples,
// two complex grids of nc samples (256 MB each at most), S(q, t) and as much
// again for the work area of its transform.  Available is what is free and
// what the handle holds for this very purpose, so that a call repeated is the
// same call.
inline DssfRoute dssf_route(bool one_workgroup, size_t n_t, size_t grid, size_t row, size_t free_bytes, size_t held) {
    const size_t avail = free_bytes + held;
    const size_t nc = std::max<size_t>(1, std::min(n_t, (size_t(256) << 20) / (grid * 16)));
    const size_t samples = 8 * n_t * grid, all = samples + 32 * nc * grid + 32 * n_t * row;
    if (!one_workgroup || samples > avail / 4 || all > avail / 4 * 3) return {false, 1};
    return {true, nc};
}

}  // namespace cslh
