// csl_record.hpp — wave sums of several values at once and the LDS barrier,
// shared by the persistent kernels (csl_trajectory.hip, csl_mixed_waves.hip,
// csl_mixed_persist.hip).
#pragma once

#include "csl_lds.hpp"

namespace csl {

namespace {

// Orders the LDS accesses of the workgroup: what __syncthreads does without
// waiting for global stores (the records' own stores stay in flight).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// v + w with the upper half of the wave taken from the partner operand:
// lanes 0..31 hold v summed over the two halves, lanes 32..63 w.
__device__ __forceinline__ double fold_halves(double v, double w) {
    auto lo = __builtin_amdgcn_permlane32_swap(unsigned(__double2loint(v)), unsigned(__double2loint(w)), false, false);
    auto hi = __builtin_amdgcn_permlane32_swap(unsigned(__double2hiint(v)), unsigned(__double2hiint(w)), false, false);
    return __hiloint2double(int(hi[0]), int(lo[0])) + __hiloint2double(int(hi[1]), int(lo[1]));
}

// The same between neighbouring rows of 16 lanes: even rows v, odd rows w.
__device__ __forceinline__ double fold_rows(double v, double w) {
    auto lo = __builtin_amdgcn_permlane16_swap(unsigned(__double2loint(v)), unsigned(__double2loint(w)), false, false);
    auto hi = __builtin_amdgcn_permlane16_swap(unsigned(__double2hiint(v)), unsigned(__double2hiint(w)), false, false);
    return __hiloint2double(int(hi[0]), int(lo[0])) + __hiloint2double(int(hi[1]), int(lo[1]));
}

// Sum over the 16 lanes of a row, in every lane of the row.
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_f64<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
    v += dpp_f64<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
    v += dpp_f64<0x124, 0xf>(v);  // row_ror:4
    v += dpp_f64<0x128, 0xf>(v);  // row_ror:8
    return v;
}

// Sums of four values over the wave, stored to out[0..3]: 21 instructions
// instead of 72 for four separate wave sums.  All lanes must be active.
__device__ __forceinline__ void wave_sum4(double a, double b, double c, double d, int lane, double* out) {
    const double v = row_sum(fold_rows(fold_halves(a, b), fold_halves(c, d)));
    // rows hold a, c, b, d
    if ((lane & 15) == 0) {
        const int r = lane >> 4;
        out[(r & 1) << 1 | r >> 1] = v;
    }
}

}  // namespace

}  // namespace csl
