// csl_mixed_waves.hip — persistent batched RK4 kernel of small mixed SU(2) +
// SU(3) lattices: one workgroup per trajectory (or piece of the work split),
// one wave per unit of 64 sites of one species, both species' waves running
// side by side.
//
// The stage values of both species (3 and 8 components) fit LDS twice, so a
// stage is one gather, the field, the update, one store and one barrier; x,
// the accumulator and the site's own stage value stay in VGPRs.  Against the
// kernel of the larger lattices (csl_mixed_persist.hip: SU(2) sites, barrier,
// SU(3) sites in place, barrier, store, barrier, with x and two components
// in global memory) a stage of the 4x4x4 TmFeO3-like cell has the waves of
// one phase on all four SIMDs instead of two phases of four waves each.
//
// What bounds it: the chain of one wave's stage (about 290 FP64 instructions
// of an SU(3) site with eight Fe-Tm bonds) with two to four waves per SIMD:
// 2.2 us a stage of that cell, 13.5 on the other kernel before.
// The constant part of the fields, the pulse envelopes and the records are
// handled as in csl_trajectory.hip, kChunk steps at a time.
#include <algorithm>
#include <type_traits>

#include "csl_mixed_lds.hpp"

namespace csl {

namespace {

constexpr int kChunk = 4;   // steps whose records and envelopes go together

// LDS layout (in doubles)
struct Lay {
    // stage values of one buffer: SU(2) [NP2 + 1][3], SU(3) [NP3 + 1][6] and
    // [NP3 + 1][2]; the last record of each is zero (csl_mixed_pack.hpp)
    int f, t, t2;
    int buf;                 // size of a buffer
    int cst, hin, drv, red;  // per-sublattice B, d0, d1; field rows; envelopes; record sums
    int rows, width;         // 3 A2 + 8 A3; sums per unit and record
    int total;
    __host__ __device__ Lay(int NP2, int NP3, int A2, int A3, int nwaves) {
        t = 0;
        t2 = 6 * (NP3 + 1);
        f = 8 * (NP3 + 1);
        buf = f + 3 * (NP2 + 1);
        buf += buf & 1;
        rows = 3 * A2 + 8 * A3;
        width = (A3 & 1) ? 20 : 12;
        cst = 2 * buf;
        hin = cst + 3 * rows;
        drv = hin + 8 * rows;
        red = drv + 2 * kChunk * 12;
        red += red & 1;
        total = red + kChunk * nwaves * width;
    }
};

// The per-site arithmetic of one species: D components, its field from the
// stage values at `buf`, and its derivative.
template <int Z22, int ZM>
struct Fe {
    static constexpr int D = 3;
    int q22[8], q23[8];
    __device__ __forceinline__ void partners(const MixDev* M, int p) {
        unpack8(M->q22[p], q22);
        unpack8(M->q23[p], q23);
    }
    __device__ __forceinline__ void field(cptr<MixDev> M, const Lay& Y, const double* buf, int a, int, const double* S,
                                          double H[3]) const {
        if (M->has_onsite2) {
            const cptr<double> A2 = as_const(M->onsite2) + a * 9;
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int e = 0; e < 3; ++e) H[d] = fma(A2[d * 3 + e], S[e], H[d]);
        }
        const cptr<double> J2 = as_const(M->jpad) + M->j22off + a * (Z22 * 9);
#pragma unroll
        for (int k = 0; k < Z22; ++k) {
            double s[3];
            ld3(buf + Y.f + 3 * q22[k], s);
#pragma unroll
            for (int e = 0; e < 3; ++e)
#pragma unroll
                for (int d = 0; d < 3; ++d) H[d] = fma(J2[k * 9 + d * 3 + e], s[e], H[d]);
        }
        const cptr<double> J3 = as_const(M->jpad) + a * (ZM * 24);
#pragma unroll
        for (int k = 0; k < ZM; ++k) {
            double s[8];
            ld8(buf + Y.t + 6 * q23[k], buf + Y.t2 + 2 * q23[k], s);
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int d = 0; d < 3; ++d) H[d] = fma(J3[k * 24 + d * 8 + e], s[e], H[d]);
        }
    }
    __device__ __forceinline__ void rhs(cptr<MixDev> M, int, bool, const double* H, const double* S, double k[3]) const {
        ll_mixed_su2(H, S, M->alpha, k);
    }
    static __device__ __forceinline__ void load(const Lay& Y, const double* buf, int p, double v[3]) {
        ld3(buf + Y.f + 3 * p, v);
    }
    static __device__ __forceinline__ void store(const Lay& Y, double* buf, int p, const double v[3]) {
        double* r = buf + Y.f + 3 * p;
        r[0] = v[0];
        r[1] = v[1];
        r[2] = v[2];
    }
};

template <int ZM, bool TT>
struct Tm {
    static constexpr int D = 8;
    int q32[8], q33[4];
    __device__ __forceinline__ void partners(const MixDev* M, int p) {
        unpack8(M->q32[p], q32);
        if constexpr (TT) {
            const uint2 v = M->q33[p];
            q33[0] = lo16(v.x);
            q33[1] = hi16(v.x);
            q33[2] = lo16(v.y);
            q33[3] = hi16(v.y);
        }
    }
    __device__ __forceinline__ void field(cptr<MixDev> M, const Lay& Y, const double* buf, int a, int, const double* S,
                                          double H[8]) const {
        if (M->has_onsite3) {
            const cptr<double> A3 = as_const(M->onsite3) + a * 64;
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int e = 0; e < 8; ++e) H[d] = fma(A3[d * 8 + e], S[e], H[d]);
        }
        if constexpr (TT) {
            const int c33 = uniform(as_const(M->e33.cnt_atom)[a]);
#pragma unroll
            for (int k = 0; k < kMixZ33; ++k) {
                if (k < c33) {
                    double s[8];
                    ld8(buf + Y.t + 6 * q33[k], buf + Y.t2 + 2 * q33[k], s);
                    const cptr<double> J = as_const(M->e33.mats) + (a * M->e33.zmax + k) * 64;
#pragma unroll
                    for (int d = 0; d < 8; ++d)
#pragma unroll
                        for (int e = 0; e < 8; ++e) H[d] = fma(J[d * 8 + e], s[e], H[d]);
                }
            }
        }
        const cptr<int> off = as_const(M->j32pad) + a * ZM;
#pragma unroll
        for (int k = 0; k < ZM; ++k) {
            double s[3];
            ld3(buf + Y.f + 3 * q32[k], s);
            const cptr<double> J = as_const(M->jpad) + uniform(off[k]);
#pragma unroll
            for (int e = 0; e < 3; ++e)
#pragma unroll
                for (int d = 0; d < 8; ++d) H[d] = fma(J[e * 8 + d], s[e], H[d]);
        }
    }
    __device__ __forceinline__ void rhs(cptr<MixDev> M, int p, bool real, const double* H, const double* S,
                                        double k[8]) const {
        su3_cross(H, S, k);
        if (M->has_bloch && real) {  // mixed_lattice_md.cpp:596-605
#pragma unroll
            for (int d = 0; d < 8; ++d)
                if (M->gamma[d] != 0.0) k[d] -= M->gamma[d] * (S[d] - M->eq3[size_t(d) * M->NP3 + p]);
        }
    }
    static __device__ __forceinline__ void load(const Lay& Y, const double* buf, int p, double v[8]) {
        ld8(buf + Y.t + 6 * p, buf + Y.t2 + 2 * p, v);
    }
    static __device__ __forceinline__ void store(const Lay& Y, double* buf, int p, const double v[8]) {
        st8(buf + Y.t + 6 * p, buf + Y.t2 + 2 * p, v);
    }
};

// All pieces of the workgroup for a wave of species SP (its unit `u`); the
// barriers of the two species' waves pair up by count.
template <class SP>
__device__ __forceinline__ void run_unit(const MixKernArgs& K, double* smem, const Lay& Y, int wave, int nwaves, int u) {
    constexpr int D = SP::D;
    constexpr bool FE = D == 3;
    const MixDev* const Mg = K.M;
    const cptr<MixDev> M0 = as_const(Mg);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), T = nwaves * kWave;
    const int NP2 = M0->NP2, NP3 = M0->NP3, A2 = M0->A2, A3 = M0->A3, npad = M0->npad;
    const int NP = FE ? NP2 : NP3;
    const int p = u * kWave + lane;
    const int a = uniform(u * kWave / npad);
    const bool real = p - a * npad < M0->n_cells;
    const int row0 = FE ? 3 * a : 3 * A2 + 8 * a;      // this sublattice's rows of cst / hin
    const size_t SZ = 3 * size_t(NP2) + 8 * size_t(NP3);
    const size_t xo = FE ? 0 : 3 * size_t(NP2);
    const MixTables Q{smem + Y.cst, smem + Y.hin, smem + Y.drv, smem + Y.red, Y.rows};
    const int R = Y.rows, W = Y.width;
    SP sp;
    sp.partners(Mg, p);
    const double dt = K.A.dt;
    const double b16 = (1.0 / 6.0) * dt, b13 = (1.0 / 3.0) * dt;

    MixPiece P;
    for (int piece = 0; mix_piece(K.A, piece, P); ++piece) {
        const int b = P.b, s_begin = P.s_begin, s_end = P.s_end;
        double* const X = K.A.X + size_t(b) * SZ + xo;
        const bool drive = K.A.tp != nullptr;
        if (P.wait >= 0) mix_wait_seam(K.A, P.wait, tid);
        __syncthreads();  // the previous piece is done with the LDS
        // padding lanes hold zeros and gather zeros: their derivative is zero
        if (tid < 22) {
            double* b0 = smem + tid / 11 * Y.buf;
            const int i = tid % 11;
            b0[i < 6 ? Y.t + 6 * NP3 + i : (i < 8 ? Y.t2 + 2 * NP3 + i - 6 : Y.f + 3 * NP2 + i - 8)] = 0.0;
        }
        double x[D], acc[D], y[D];
#pragma unroll
        for (int d = 0; d < D; ++d) x[d] = real ? X[size_t(d) * NP + p] : 0.0;
        SP::store(Y, smem, p, x);
        mix_fill_tables(M0, Q, tid, T);
        __syncthreads();

        // envelopes by the last wave
        auto write_drive = [&](int n0, int cp) {
            if (drive && wave == nwaves - 1) mix_write_drive(Q, b, n0, s_end, cp, kChunk, lane);
        };
        auto write_hin = [&](const double* f, int par) {
            if (drive) mix_write_hin(Q, f, par, 3 * A2, tid, T);
        };
        write_drive(s_begin, 0);
        lds_barrier();
        write_hin(Q.drv, 0);
        lds_barrier();

        // this unit's sums of S (and the sign-alternating ones when the sign
        // changes from cell to cell) and of its share of the energy
        auto reduce_obs = [&](int slot, const double* S, double e) {
            double* r = Q.red + (slot * nwaves + wave) * W;
            wave_sum4(S[0], S[1], S[2], e, lane, r);
            if constexpr (!FE) {
                wave_sum4(S[3], S[4], S[5], S[6], lane, r + 4);
                wave_sum4(S[7], 0.0, 0.0, 0.0, lane, r + 8);
                if (A3 & 1) {
                    const double sg = (((p - a * npad) * A3 + a) & 1) ? -1.0 : 1.0;
                    wave_sum4(sg * S[0], sg * S[1], sg * S[2], sg * S[3], lane, r + 12);
                    wave_sum4(sg * S[4], sg * S[5], sg * S[6], sg * S[7], lane, r + 16);
                }
            }
        };
        // records ri0 .. ri0 + cnt - 1, one wave each
        auto publish = [&](int ri0, int cnt) {
            for (int k = wave; k < cnt; k += nwaves) {
                const double *r2 = Q.red + k * nwaves * W, *r3 = r2 + (NP2 / kWave) * W;
                mix_publish(
                    b, ri0 + k, lane, [&](int w, int c) { return r2[w * W + c]; },
                    [&](int w, int c) { return r3[w * W + (c < 3 ? c : c + 1)]; },
                    [&](int w, int c) { return r3[w * W + 12 + c]; },
                    [&] {
                        double e = 0.0;
                        for (int w = 0; w < nwaves; ++w) e += r2[w * W + 3];
                        return e;
                    });
            }
        };

        auto stage = [&](auto s_, int par, int slot) {
            constexpr int s = decltype(s_)::value;
            constexpr int st = s == 0 ? 3 : (s == 3 ? 2 : 1);
            const double cdt = s == 2 ? dt : 0.5 * dt;
            const double bdt = (s == 0 || s == 3) ? b16 : b13;
            const cptr<MixDev> M = as_const(Mg) + opaque_zero();
            const double* cur = smem + (s & 1) * Y.buf;
            double* nxt = smem + (1 - (s & 1)) * Y.buf;
            const double* S = s == 0 ? x : y;
            const double* h = Q.hin + (par * 4 + st) * R + row0;
            double H[D];
#pragma unroll
            for (int d = 0; d < D; ++d) H[d] = h[d];
            sp.field(M, Y, cur, a, p, S, H);
            if (s == 0 && slot >= 0) {
                // S.(H - B) of the undriven field: twice the energy
                double e = 0.0;
#pragma unroll
                for (int d = 0; d < D; ++d) e = fma(S[d], H[d] + h[d], e);
                reduce_obs(slot, S, e);
            }
            if constexpr (s == 0) {
                // the drive after the record (a driven field would round at the drive's size)
                const double* dr = Q.hin + par * 4 * R + row0;
#pragma unroll
                for (int d = 0; d < D; ++d) H[d] -= dr[d];
            }
            double k[D];
            sp.rhs(M, p, real, H, S, k);
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (s == 0) acc[d] = x[d] + bdt * k[d];
                else if (s < 3) acc[d] = acc[d] + bdt * k[d];
                else x[d] = acc[d] + bdt * k[d];
                if (s < 3) y[d] = x[d] + cdt * k[d];
            }
            SP::store(Y, nxt, p, s < 3 ? y : x);
            lds_barrier();
        };

        const int si = K.A.save_interval;
        int ri = (s_begin + si - 1) / si, next_rec = ri * si;
        for (int n0 = s_begin, cp = 0; n0 < s_end; n0 += kChunk, cp ^= 1) {
            const int n1 = min(n0 + kChunk, s_end);
            const int ri0 = ri;
            write_drive(n1, cp ^ 1);
            for (int n = n0; n < n1; ++n) {
                const int par = (n - s_begin) & 1;
                int slot = -1;
                if (n == next_rec) {
                    slot = ri - ri0;
                    ++ri;
                    next_rec += si;
                }
                const int q = n + 1 - n0;
                if (n + 1 < s_end && q < kChunk) write_hin(Q.drv + (cp * kChunk + q) * 12, par ^ 1);
                stage(std::integral_constant<int, 0>{}, par, slot);
                if (n + 1 == n1 && ri > ri0) publish(ri0, ri - ri0);
                stage(std::integral_constant<int, 1>{}, par, -1);
                // the next chunk's envelopes are complete since stage 0
                if (n + 1 < s_end && q == kChunk) write_hin(Q.drv + (cp ^ 1) * kChunk * 12, par ^ 1);
                stage(std::integral_constant<int, 2>{}, par, -1);
                stage(std::integral_constant<int, 3>{}, par, -1);
            }
        }

        const MixArgsP G = mix_kern_args();
        // x back to its slot: the final state, or the seam's
        if (real) {
#pragma unroll
            for (int d = 0; d < D; ++d) X[size_t(d) * NP + p] = x[d];
        }
        if (P.post >= 0) {
            __threadfence();
            __syncthreads();
            if (tid == 0) __hip_atomic_store(G->A.flags + P.post, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (s_end == G->A.n_steps) {
            // final record: the state after the last step (buffer 0), undriven
            double H[D], e = 0.0;
#pragma unroll
            for (int d = 0; d < D; ++d) H[d] = -Q.cst[3 * (row0 + d)];
            sp.field(as_const(Mg) + opaque_zero(), Y, smem, a, p, x, H);
#pragma unroll
            for (int d = 0; d < D; ++d) e = fma(x[d], H[d] - Q.cst[3 * (row0 + d)], e);
            reduce_obs(0, x, e);
            lds_barrier();
            publish(G->A.n_rec - 1, 1);
        }
    }
}

}  // namespace

template <int T, int Z22, int ZM, bool TT>
__global__ void __launch_bounds__(T) k_mixed_waves(MixKernArgs K) {
    extern __shared__ double smem[];
    const cptr<MixDev> M = as_const(K.M);
    const int nwaves = int(blockDim.x) >> 6;
    const int wave = uniform(threadIdx.x >> 6);
    const Lay Y(M->NP2, M->NP3, M->A2, M->A3, nwaves);
    const int nu2 = M->NP2 / kWave;
    if (wave < nu2) run_unit<Fe<Z22, ZM>>(K, smem, Y, wave, nwaves, wave);
    else run_unit<Tm<ZM, TT>>(K, smem, Y, wave, nwaves, wave - nu2);
}

namespace {

template <int T, int Z22, int ZM, bool TT>
hipError_t launch_w(const MixDev* M, const MixPersistArgs& A, int block, int grid, size_t lds, hipStream_t st, int* occ) {
    auto kern = k_mixed_waves<T, Z22, ZM, TT>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, kern, block, lds);
    const MixKernArgs K{M, A};
    hipLaunchKernelGGL(kern, dim3(unsigned(grid)), dim3(unsigned(block)), lds, st, K);
    return hipGetLastError();
}

template <int T>
hipError_t launch_w_z(const MixDev& Mh, bool tt, const MixDev* M, const MixPersistArgs& A, int block, int grid,
                      size_t lds, hipStream_t st, int* occ) {
    const int z = Mh.jz22 * 10 + Mh.jzm;
    if (tt) return z == 88 ? launch_w<T, 8, 8, true>(M, A, block, grid, lds, st, occ) : hipErrorInvalidValue;
    switch (z) {
        case 64: return launch_w<T, 6, 4, false>(M, A, block, grid, lds, st, occ);
        case 68: return launch_w<T, 6, 8, false>(M, A, block, grid, lds, st, occ);
        case 84: return launch_w<T, 8, 4, false>(M, A, block, grid, lds, st, occ);
        case 88: return launch_w<T, 8, 8, false>(M, A, block, grid, lds, st, occ);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

size_t mixed_waves_lds_bytes(const MixDev& M) {
    return sizeof(double) * size_t(Lay(M.NP2, M.NP3, M.A2, M.A3, (M.NP2 + M.NP3) / kWave).total);
}

hipError_t launch_mixed_waves(const MixDev& Mh, const MixDev* M, const MixPersistArgs& A, const MixPersistShape& sh,
                              int grid, hipStream_t st, int* occ) {
    const size_t lds = mixed_waves_lds_bytes(Mh);
    // up to eight waves may use 256 VGPRs each
    return sh.block <= 512 ? launch_w_z<512>(Mh, sh.tt, M, A, sh.block, grid, lds, st, occ)
                           : launch_w_z<1024>(Mh, sh.tt, M, A, sh.block, grid, lds, st, occ);
}

}  // namespace csl
