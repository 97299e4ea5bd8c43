// csl_mixed_persist.hip — persistent batched RK4 kernel of the mixed
// SU(2) + SU(3) lattice: one workgroup integrates one trajectory (or a piece
// of one) for the whole time grid (mixed_lattice_gpu.cu:278-347 launches one
// kernel per RK stage instead), so the per-stage state never crosses HBM.
// Lattices of at most 16 units of 64 sites run on csl_mixed_waves.hip.
//
// On-chip budget of one trajectory of the 8x8x8 TmFeO3-like cell (2048 SU(2)
// + 2048 SU(3) sites, 176 KB of stage values): RK4 needs the step-start
// state x, the accumulator and the stage values.  The stage values are what
// the neighbours gather, so they go to LDS: the SU(2) sites as records of 24
// bytes, the SU(3) components 0..5 as records of 48 bytes (three 16-byte
// loads at one address; the strides spread a wave's records over all banks).
// SU(3) components 6 and 7 go to LDS too where they fit (GLDS, up to 1536
// sites of each species) and otherwise to a per-workgroup global buffer with
// two parities that stays in L2, one 16-byte access per site.  The
// accumulators of a thread's sites live in VGPRs; x lives in the trajectory's
// own slot of the global state array (read in stages 1 and 2, written in
// stage 3).
//
// Per stage without SU(3)-SU(3) bonds: the SU(2) sites from y_s, their next
// values kept in VGPRs -> barrier -> the SU(3) sites, updated in place (only
// the owner reads an SU(3) site's own value then) -> barrier -> the SU(2)
// next values into LDS -> barrier.  With them (TT) both species' next values
// are held until one barrier.  A wave owns SPT consecutive units of 64 sites
// of each species and advances them one by one (two of one sublattice
// together, their bond matrices fetched once, spilled: 33.5 against 28.5 us
// a stage of the 8x8x8 cell).
//
// Field rows, pulse envelopes and records are handled as in
// csl_trajectory.hip: field rows from LDS, envelopes of two steps
// at a time, records from the waves' sums of S and S.H, two at a time; lattices
// with many sublattices keep smaller tables (TIGHT, csl_mixed_lay.hpp).  With
// every record's 33 wave sums in shuffles, an envelope evaluation per wave
// and stage, one 4-byte partner load per bond and one 8-byte access per
// component a stage of the 8x8x8 cell took 36.8 us; it takes 27 (0.28 of the
// SIMD cycles issue FP64 work, 0.42 anything; x from global memory costs 3.6
// us; 5.4 TB/s of x, components 6 and 7 and partner words leave the L2s).
#include <algorithm>
#include <type_traits>

#include "csl_mixed_lay.hpp"
#include "csl_mixed_lds.hpp"

namespace csl {

namespace {

using Lay = MixPersistLay;

template <int Z22, int ZM, bool GLDS>
struct Field {
    const MixDev* Mg;
    const double* smem;
    const Lay& Y;
    const double2* g;        // components 6, 7 of the stage (global), !GLDS

    __device__ __forceinline__ void tm(int q, double v[8]) const {
        const double2* r = reinterpret_cast<const double2*>(smem + Y.t + 6 * q);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double2 a = r[i];
            v[2 * i] = a.x;
            v[2 * i + 1] = a.y;
        }
        const double2 a = GLDS ? *reinterpret_cast<const double2*>(smem + Y.t2 + 2 * q) : g[q];
        v[6] = a.x;
        v[7] = a.y;
    }

    // field of SU(2) site p of sublattice a.  The bonds are kept apart (an
    // opaque address each, end_bond): the compiler otherwise loads every
    // bond's matrix at once and spills them
    __device__ __forceinline__ void fe(int a, int p, const double S[3], double (&H)[3]) const {
        const cptr<MixDev> M = as_const(Mg) + opaque_zero();
        int q22[8], q23[8];
        unpack8(M->q23[p], q23);
        unpack8(M->q22[p], q22);
        // components 6 and 7 of the next kAhead SU(3) partners are on their
        // way from global memory (L2), the first ones while the SU(2) bonds run
        constexpr int kAhead = GLDS ? 1 : 4;
        double2 gl[kAhead];
        if constexpr (!GLDS) {
#pragma unroll
            for (int k = 0; k < kAhead; ++k) gl[k] = g[q23[k]];
        }
        if (M->has_onsite2) {
            const cptr<double> A2 = as_const(M->onsite2) + a * 9;
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int e = 0; e < 3; ++e) H[d] = fma(A2[d * 3 + e], S[e], H[d]);
        }
        const cptr<double> jp = as_const(M->jpad);
        const int j2 = M->j22off + a * (Z22 * 9), j3 = a * (ZM * 24);
#pragma unroll
        for (int k = 0; k < Z22; ++k) {
            const cptr<double> J = jp + j2 + k * 9 + opaque_zero();
            double s[3];
            ld3(smem + Y.f + 3 * q22[k], s);
#pragma unroll
            for (int e = 0; e < 3; ++e)
#pragma unroll
                for (int d = 0; d < 3; ++d) H[d] = fma(J[d * 3 + e], s[e], H[d]);
            end_bond(H);
        }
#pragma unroll
        for (int k = 0; k < ZM; ++k) {
            const cptr<double> J = jp + j3 + k * 24 + opaque_zero();
            double s[8];
            const double2* r = reinterpret_cast<const double2*>(smem + Y.t + 6 * q23[k]);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double2 v = r[i];
                s[2 * i] = v.x;
                s[2 * i + 1] = v.y;
            }
            const double2 v = GLDS ? *reinterpret_cast<const double2*>(smem + Y.t2 + 2 * q23[k]) : gl[GLDS ? 0 : k % kAhead];
            if constexpr (!GLDS)
                if (k + kAhead < ZM) gl[k % kAhead] = g[q23[k + kAhead]];
            s[6] = v.x;
            s[7] = v.y;
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int d = 0; d < 3; ++d) H[d] = fma(J[d * 8 + e], s[e], H[d]);
            end_bond(H);
        }
    }

    // bond field of SU(3) site p of sublattice a (the on-site part apart)
    template <bool TT>
    __device__ __forceinline__ void tm_bonds(int a, int p, double (&H)[8]) const {
        const cptr<MixDev> M = as_const(Mg) + opaque_zero();
        int q32[8], off[ZM];
        unpack8(M->q32[p], q32);
#pragma unroll
        for (int k = 0; k < ZM; ++k) off[k] = (as_const(M->j32pad) + a * ZM)[k];
        const cptr<double> jp = as_const(M->jpad);
        if constexpr (TT) {
            const int c33 = uniform(as_const(M->e33.cnt_atom)[a]);
            const uint2 v = M->q33[p];
            const int q33[4] = {lo16(v.x), hi16(v.x), lo16(v.y), hi16(v.y)};
#pragma unroll
            for (int k = 0; k < kMixZ33; ++k) {
                if (k < c33) {
                    double s[8];
                    tm(q33[k], s);
                    const cptr<double> J = as_const(M->e33.mats) + (a * M->e33.zmax + k) * 64;
#pragma unroll
                    for (int d = 0; d < 8; ++d)
#pragma unroll
                        for (int e = 0; e < 8; ++e) H[d] = fma(J[d * 8 + e], s[e], H[d]);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < ZM; ++k) {
            const cptr<double> J = jp + uniform(off[k]) + opaque_zero();
            double s[3];
            ld3(smem + Y.f + 3 * q32[k], s);
#pragma unroll
            for (int e = 0; e < 3; ++e)
#pragma unroll
                for (int d = 0; d < 8; ++d) H[d] = fma(J[e * 8 + d], s[e], H[d]);
            end_bond(H);
        }
    }
};

}  // namespace

template <int SPT, int T, int Z22, int ZM, bool TT, bool GLDS, bool TIGHT>
__global__ void __launch_bounds__(T) k_mixed_persist(MixKernArgs K) {
    extern __shared__ double smem[];
    constexpr int nwaves = T / kWave;
    const MixDev* const Mg = K.M;
    const cptr<MixDev> M0 = as_const(Mg);
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = uniform(tid >> 6);
    const int NP2 = M0->NP2, NP3 = M0->NP3, A2 = M0->A2, A3 = M0->A3, npad = M0->npad, n_cells = M0->n_cells;
    const Lay Y(NP2, NP3, A2, A3, nwaves, GLDS, TIGHT);
    constexpr int kChunk = TIGHT ? 1 : 2;
    const MixTables Q{smem + Y.cst, smem + Y.hin, smem + Y.drv, smem + Y.red, Y.rows};
    const int R = Y.rows;
    const int GS = NP3 + 1;                          // a parity of components 6, 7 in global memory
    double2* const Gw = GLDS ? nullptr : reinterpret_cast<double2*>(K.A.G) + size_t(blockIdx.x) * 2 * size_t(GS);
    const size_t SZ = 3 * size_t(NP2) + 8 * size_t(NP3);
    const size_t o3 = 3 * size_t(NP2);
    const double dt = K.A.dt;
    const bool drive = K.A.tp != nullptr;
    const int u0 = wave * SPT;                       // first unit of the wave (both species)
    const int p0 = u0 * kWave + lane;
    const int m2 = min(max(Y.n2 - u0, 0), SPT), m3 = min(max(Y.n3 - u0, 0), SPT);  // its units
    auto atom = [&](int j) { return uniform((u0 + j) * kWave / npad); };
    auto real = [&](int j) { const int p = p0 + j * kWave; return p - p / npad * npad < n_cells; };

    MixPiece P;
    for (int piece = 0; mix_piece(K.A, piece, P); ++piece) {
        const int b = P.b, s_begin = P.s_begin, s_end = P.s_end;
        double* const X = K.A.X + size_t(b) * SZ;
        if (P.wait >= 0) mix_wait_seam(K.A, P.wait, tid);
        __syncthreads();  // the previous piece is done with LDS and G
        // initial state: the stage values of stage 0; padding lanes hold
        // zeros and gather zeros, so their derivative is zero
        if (tid < 6) smem[Y.t + 6 * NP3 + tid] = 0.0;
        if (tid < 3) smem[Y.f + 3 * NP2 + tid] = 0.0;
        if (tid < 2) {
            if constexpr (GLDS) smem[Y.t2 + 2 * NP3 + tid] = 0.0;
            else Gw[tid * GS + NP3] = make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            const int p = p0 + j * kWave;
            if (j < m2) {
                double* r = smem + Y.f + 3 * p;
                const bool ok = real(j);
#pragma unroll
                for (int c = 0; c < 3; ++c) r[c] = ok ? X[size_t(c) * NP2 + p] : 0.0;
            }
            if (j < m3) {
                const bool ok = real(j);
                double v[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) v[c] = ok ? X[o3 + size_t(c) * NP3 + p] : 0.0;
                double2* r = reinterpret_cast<double2*>(smem + Y.t + 6 * p);
#pragma unroll
                for (int i = 0; i < 3; ++i) r[i] = make_double2(v[2 * i], v[2 * i + 1]);
                if constexpr (GLDS) *reinterpret_cast<double2*>(smem + Y.t2 + 2 * p) = make_double2(v[6], v[7]);
                else Gw[p] = make_double2(v[6], v[7]);
            }
        }
        if constexpr (TIGHT)
            for (int st = 0; st < 4; ++st) mix_write_row(M0, Q, nullptr, st, 3 * A2, tid, T);
        else
            mix_fill_tables(M0, Q, tid, T);
        __syncthreads();
        auto write_drive = [&](int n0, int cp) {
            if (drive && wave == nwaves - 1) mix_write_drive(Q, b, n0, s_end, cp, kChunk, lane);
        };
        auto write_hin = [&](const double* f, int par) {
            if (!drive) return;
            if constexpr (TIGHT)
                for (int st = 0; st < 3; ++st) mix_write_row(M0, Q, f, st, 3 * A2, tid, T);
            else
                mix_write_hin(Q, f, par, 3 * A2, tid, T);
        };
        // TIGHT: the rows of the step before are replaced one by one as they
        // have been read: 0 by stage 0, 1 by stage 2, 2 by stage 3 (its
        // successor is written in stage 1 of its own step)
        auto replace_rows = [&](int s, const double* f, const double* f_next, bool more) {
            if (!drive) return;
            if (s == 1) mix_write_row(M0, Q, f, 2, 3 * A2, tid, T);
            if (s == 2 && more) mix_write_row(M0, Q, f_next, 0, 3 * A2, tid, T);
            if (s == 3 && more) mix_write_row(M0, Q, f_next, 1, 3 * A2, tid, T);
        };
        auto field_b = [&](int i) { return TIGHT ? mix_row(M0, i).B : Q.cst[3 * i]; };
        write_drive(s_begin, 0);
        lds_barrier();
        write_hin(Q.drv, 0);
        lds_barrier();

        auto publish = [&](int ri0, int cnt) {
            for (int k = wave; k < cnt; k += nwaves) {
                const double *r2 = Q.red + k * Y.rec, *r3 = r2 + 4 * Y.n2, *ra = r3 + 8 * Y.n3;
                const double* re = r2 + Y.rec - 4 * nwaves;
                mix_publish(
                    b, ri0 + k, lane, [&](int w, int c) { return r2[w * 4 + c]; },
                    [&](int w, int c) { return r3[w * 8 + c]; }, [&](int w, int c) { return ra[w * 8 + c]; },
                    [&] {
                        double e = 0.0;
                        for (int w = 0; w < nwaves; ++w) e += re[w * 4];
                        return e;
                    });
            }
        };
        // sums of an SU(2) / SU(3) unit's stage values into record `slot`
        auto sums2 = [&](int slot, int j, const double S[3]) {
            wave_sum4(S[0], S[1], S[2], 0.0, lane, Q.red + slot * Y.rec + 4 * (u0 + j));
        };
        auto sums3 = [&](int slot, int j, const double S[8]) {
            double* r = Q.red + slot * Y.rec + 4 * Y.n2 + 8 * (u0 + j);
            wave_sum4(S[0], S[1], S[2], S[3], lane, r);
            wave_sum4(S[4], S[5], S[6], S[7], lane, r + 4);
            if (A3 & 1) {
                const int p = p0 + j * kWave, a = atom(j);
                const double sg = (((p - a * npad) * A3 + a) & 1) ? -1.0 : 1.0;
                r += 8 * Y.n3;
                wave_sum4(sg * S[0], sg * S[1], sg * S[2], sg * S[3], lane, r);
                wave_sum4(sg * S[4], sg * S[5], sg * S[6], sg * S[7], lane, r + 4);
            }
        };
        auto sum_e = [&](int slot, double e) {
            wave_sum4(e, 0.0, 0.0, 0.0, lane, Q.red + slot * Y.rec + (Y.rec - 4 * nwaves) + 4 * wave);
        };

        double acc2[SPT][3], acc3[SPT][8];
        // One RK4 stage (runtime index s).  slot >= 0 in stage 0 of a
        // recorded step.
        auto stage = [&](int s, int par, int slot) __attribute__((always_inline)) {
            const double cdt = s == 2 ? dt : 0.5 * dt;
            const double bdt = (s == 0 || s == 3) ? (1.0 / 6.0) * dt : (1.0 / 3.0) * dt;
            const int set = TIGHT ? 0 : par * 4;
            const double* hrow = Q.hin + (set + (s == 0 ? 3 : (s == 3 ? 2 : 1))) * R;
            const double* drow = Q.hin + set * R;   // stage 0: the drive, after the record's undriven energy
            const Field<Z22, ZM, GLDS> F{Mg, smem, Y, GLDS ? nullptr : Gw + (s & 1) * GS};
            double2* const Gn = GLDS ? nullptr : Gw + (1 - (s & 1)) * GS;
            double e = 0.0;
            double y2[SPT][3];
            auto fe_unit = [&](int j) __attribute__((always_inline)) {
                const int p = p0 + j * kWave, a = atom(j);
                const cptr<MixDev> M = as_const(Mg) + opaque_zero();
                double S[3], H[3], xv[3];
                ld3(smem + Y.f + 3 * p, S);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    H[d] = hrow[3 * a + d];
                    // x in flight while the bonds run
                    xv[d] = (s == 1 || s == 2) ? X[size_t(d) * NP2 + p] : S[d];
                }
                F.fe(a, p, S, H);
                if (slot >= 0) {
#pragma unroll
                    for (int d = 0; d < 3; ++d) e = fma(S[d], H[d] + hrow[3 * a + d], e);
                    sums2(slot, j, S);
                }
                if (s == 0) {
#pragma unroll
                    for (int d = 0; d < 3; ++d) H[d] -= drow[3 * a + d];
                }
                double k[3];
                ll_mixed_su2(H, S, M->alpha, k);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    acc2[j][d] = (s == 0 ? S[d] : acc2[j][d]) + bdt * k[d];
                    y2[j][d] = s < 3 ? xv[d] + cdt * k[d] : acc2[j][d];
                }
                if (s == 3 && real(j)) {
#pragma unroll
                    for (int d = 0; d < 3; ++d) X[size_t(d) * NP2 + p] = y2[j][d];
                }
            };
            double y3[TT ? SPT : 1][8];
            auto tm_unit = [&](int j) __attribute__((always_inline)) {
                const int p = p0 + j * kWave, a = atom(j);
                const cptr<MixDev> M = as_const(Mg) + opaque_zero();
                const double* hr = hrow + 3 * A2 + 8 * a;
                double H[8], xv[8];
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    H[d] = hr[d];
                    xv[d] = (s == 1 || s == 2) ? X[o3 + size_t(d) * NP3 + p] : 0.0;
                }
                F.template tm_bonds<TT>(a, p, H);
                double S[8];
                F.tm(p, S);
                if (M->has_onsite3) {
                    const cptr<double> A3m = as_const(M->onsite3) + a * 64;
#pragma unroll
                    for (int d = 0; d < 8; ++d)
#pragma unroll
                        for (int c = 0; c < 8; ++c) H[d] = fma(A3m[d * 8 + c], S[c], H[d]);
                }
                if (slot >= 0) {
#pragma unroll
                    for (int d = 0; d < 8; ++d) e = fma(S[d], H[d] + hr[d], e);
                    sums3(slot, j, S);
                }
                if (s == 0) {
                    const double* dr = drow + 3 * A2 + 8 * a;
#pragma unroll
                    for (int d = 0; d < 8; ++d) H[d] -= dr[d];
                }
                double k[8];
                su3_cross(H, S, k);
                if (M->has_bloch && real(j)) {  // mixed_lattice_md.cpp:596-605
#pragma unroll
                    for (int d = 0; d < 8; ++d)
                        if (M->gamma[d] != 0.0) k[d] -= M->gamma[d] * (S[d] - M->eq3[size_t(d) * NP3 + p]);
                }
                double y[8];
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    acc3[j][d] = (s == 0 ? S[d] : acc3[j][d]) + bdt * k[d];
                    y[d] = s < 3 ? (s == 0 ? S[d] : xv[d]) + cdt * k[d] : acc3[j][d];
                }
                if (s == 3 && real(j)) {
#pragma unroll
                    for (int d = 0; d < 8; ++d) X[o3 + size_t(d) * NP3 + p] = y[d];
                }
                if constexpr (!GLDS) Gn[p] = make_double2(y[6], y[7]);
                if constexpr (TT) {
#pragma unroll
                    for (int d = 0; d < 8; ++d) y3[j][d] = y[d];
                } else {
                    double2* r = reinterpret_cast<double2*>(smem + Y.t + 6 * p);
#pragma unroll
                    for (int c = 0; c < 3; ++c) r[c] = make_double2(y[2 * c], y[2 * c + 1]);
                    if constexpr (GLDS) *reinterpret_cast<double2*>(smem + Y.t2 + 2 * p) = make_double2(y[6], y[7]);
                }
            };
#pragma unroll
            for (int j = 0; j < SPT; ++j)
                if (j < m2) fe_unit(j);
            if constexpr (TT) {
#pragma unroll
                for (int j = 0; j < SPT; ++j)
                    if (j < m3) tm_unit(j);
                if (slot >= 0) sum_e(slot, e);
                __syncthreads();  // every read of y_s is done
#pragma unroll
                for (int j = 0; j < SPT; ++j) {
                    const int p = p0 + j * kWave;
                    if (j >= m3) break;
                    double2* r = reinterpret_cast<double2*>(smem + Y.t + 6 * p);
#pragma unroll
                    for (int c = 0; c < 3; ++c) r[c] = make_double2(y3[j][2 * c], y3[j][2 * c + 1]);
                    if constexpr (GLDS)
                        *reinterpret_cast<double2*>(smem + Y.t2 + 2 * p) = make_double2(y3[j][6], y3[j][7]);
                }
            } else {
                lds_barrier();  // the SU(2) sites' reads of y_s are done
#pragma unroll
                for (int j = 0; j < SPT; ++j)
                    if (j < m3) tm_unit(j);
                if (slot >= 0) sum_e(slot, e);
                lds_barrier();  // the SU(3) sites' reads of the SU(2) stage values are done
            }
#pragma unroll
            for (int j = 0; j < SPT; ++j) {
                if (j >= m2) break;
                double* r = smem + Y.f + 3 * (p0 + j * kWave);
#pragma unroll
                for (int d = 0; d < 3; ++d) r[d] = y2[j][d];
            }
            // y_{s+1} complete; its components 6, 7 in global memory too
            if constexpr (GLDS) lds_barrier();
            else __syncthreads();
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
#pragma unroll 1
                for (int s = 0; s < 4; ++s) {
                    // rows of the next step: this parity's were last read a
                    // step ago; the next chunk's envelopes are complete since
                    // stage 0
                    if constexpr (TIGHT)
                        replace_rows(s, Q.drv + cp * 12, Q.drv + (cp ^ 1) * 12, n + 1 < s_end);
                    else if (s == 2 && n + 1 < s_end)
                        write_hin(q < kChunk ? Q.drv + (cp * kChunk + q) * 12 : Q.drv + (cp ^ 1) * kChunk * 12, par ^ 1);
                    stage(s, par, s == 0 ? slot : -1);
                    if (s == 0 && n + 1 == n1 && ri > ri0) publish(ri0, ri - ri0);
                }
            }
        }

        const MixArgsP G = mix_kern_args();
        if (P.post >= 0) {
            // hand the state at s_end (in X since the last step's stage 3)
            // to the workgroup that continues the trajectory
            __threadfence();
            __syncthreads();
            if (tid == 0) __hip_atomic_store(G->A.flags + P.post, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        // final record: the state after the last step (the stage values of
        // the next step's stage 0), undriven
        if (s_end == G->A.n_steps) {
            const Field<Z22, ZM, GLDS> F{Mg, smem, Y, GLDS ? nullptr : Gw};
            double e = 0.0;
#pragma unroll 1
            for (int j = 0; j < m2; ++j) {
                const int p = p0 + j * kWave, a = atom(j);
                double S[3], H[3];
                ld3(smem + Y.f + 3 * p, S);
#pragma unroll
                for (int d = 0; d < 3; ++d) H[d] = -field_b(3 * a + d);
                F.fe(a, p, S, H);
#pragma unroll
                for (int d = 0; d < 3; ++d) e = fma(S[d], H[d] - field_b(3 * a + d), e);
                sums2(0, j, S);
            }
#pragma unroll 1
            for (int j = 0; j < m3; ++j) {
                const int p = p0 + j * kWave, a = atom(j);
                const int c3 = 3 * A2 + 8 * a;
                double S[8], H[8];
                F.tm(p, S);
#pragma unroll
                for (int d = 0; d < 8; ++d) H[d] = -field_b(c3 + d);
                F.template tm_bonds<TT>(a, p, H);
                if (M0->has_onsite3) {
                    const cptr<double> A3m = as_const(M0->onsite3) + a * 64;
#pragma unroll
                    for (int d = 0; d < 8; ++d)
#pragma unroll
                        for (int c = 0; c < 8; ++c) H[d] = fma(A3m[d * 8 + c], S[c], H[d]);
                }
#pragma unroll
                for (int d = 0; d < 8; ++d) e = fma(S[d], H[d] - field_b(c3 + d), e);
                sums3(0, j, S);
            }
            sum_e(0, e);
            lds_barrier();
            publish(G->A.n_rec - 1, 1);
        }
    }
}

namespace {

template <int SPT, int T, int Z22, int ZM, bool TT, bool GLDS, bool TIGHT>
hipError_t launch_mp(const MixDev* M, const MixPersistArgs& A, int grid, const Lay& Y, hipStream_t st, int* occ) {
    auto kern = k_mixed_persist<SPT, T, Z22, ZM, TT, GLDS, TIGHT>;
    const size_t lds = sizeof(double) * size_t(Y.total);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, kern, T, lds);
    const MixKernArgs K{M, A};
    hipLaunchKernelGGL(kern, dim3(unsigned(grid)), dim3(T), lds, st, K);
    return hipGetLastError();
}

Lay persist_lay(const MixDev& M, int block, bool glds) {
    return mix_persist_lay(M.NP2, M.NP3, M.A2, M.A3, block / kWave, glds);
}

// Components 6 and 7 in LDS where they fit: always up to 1024 sites of each
// species (two units per wave of 512 threads, one of 1024).
Lay glds_lay(const MixDev& M, int block) { return Lay(M.NP2, M.NP3, M.A2, M.A3, block / kWave, true, false); }

template <int SPT, int T, int Z22, int ZM, bool TT>
hipError_t launch_mp_g(const MixDev& Mh, const MixDev* M, const MixPersistArgs& A, int grid, hipStream_t st, int* occ) {
    const Lay in_lds = glds_lay(Mh, T);
    if (in_lds.total <= kMixLdsDoubles) return launch_mp<SPT, T, Z22, ZM, TT, true, false>(M, A, grid, in_lds, st, occ);
    if constexpr (SPT * T > 1024) {
        const Lay Y = persist_lay(Mh, T, false);
        return Y.tight ? launch_mp<SPT, T, Z22, ZM, TT, false, true>(M, A, grid, Y, st, occ)
                       : launch_mp<SPT, T, Z22, ZM, TT, false, false>(M, A, grid, Y, st, occ);
    }
    return hipErrorInvalidValue;
}

template <int SPT>
hipError_t launch_mp_z(const MixDev& Mh, const MixDev* M, const MixPersistArgs& A, int grid, hipStream_t st, int* occ) {
    if (Mh.jzm == 4) {
        return Mh.jz22 == 6 ? launch_mp_g<SPT, 1024, 6, 4, false>(Mh, M, A, grid, st, occ)
                            : launch_mp_g<SPT, 1024, 8, 4, false>(Mh, M, A, grid, st, occ);
    }
    return Mh.jz22 == 6 ? launch_mp_g<SPT, 1024, 6, 8, false>(Mh, M, A, grid, st, occ)
                        : launch_mp_g<SPT, 1024, 8, 8, false>(Mh, M, A, grid, st, occ);
}

}  // namespace

// Without SU(3)-SU(3) bonds: 1024 threads (4 waves per SIMD) and up to two
// units of each species per wave — the SU(3) sites update in place, so a
// thread holds only its accumulators and its SU(2) sites' next values.  With
// them: 512 threads and two to four units (the SU(3) next values are held
// too).  Lattices of at most 16 units (both species together) whose stage
// values fit LDS twice take the one-unit-per-wave kernel.
MixPersistShape mixed_persist_shape(const MixDev& M, bool tt) {
    const int units = (M.NP2 + M.NP3) / kWave, np = std::max(M.NP2, M.NP3);
    if (!M.jpad) return {0, 0, tt, false};
    if (units <= 16 && mixed_waves_lds_bytes(M) <= 160 * 1024) return {units * kWave, 1, tt, true};
    MixPersistShape sh{0, 0, tt, false};
    if (!tt) {
        if (np <= 2048) sh = {1024, np <= 1024 ? 1 : 2, false, false};
    } else {
        const int spt = (np + 511) / 512;
        if (spt <= 4) sh = {512, spt, true, false};
    }
    if (sh.block && persist_lay(M, sh.block, false).total > kMixLdsDoubles) sh = {0, 0, tt, false};
    return sh;
}

int mixed_persist_variant(const MixDev& M, const MixPersistShape& sh) {
    if (!sh.block) return 0;
    if (sh.waves) return CSL_MIXED_VARIANT_PERSISTENT | CSL_MIXED_VARIANT_UNIT_WAVES;
    if (glds_lay(M, sh.block).total <= kMixLdsDoubles) return CSL_MIXED_VARIANT_PERSISTENT;
    return CSL_MIXED_VARIANT_PERSISTENT | CSL_MIXED_VARIANT_GLOBAL_67 |
           (persist_lay(M, sh.block, false).tight ? CSL_MIXED_VARIANT_TIGHT : 0);
}

hipError_t launch_mixed_persist(const MixDev& Mh, const MixDev* M, const MixPersistArgs& A, const MixPersistShape& sh,
                                int grid, hipStream_t st, int* occ) {
    if (!sh.tt && sh.block == 1024) {
        if (sh.spt == 1) return launch_mp_z<1>(Mh, M, A, grid, st, occ);
        if (sh.spt == 2) return launch_mp_z<2>(Mh, M, A, grid, st, occ);
    }
    if (sh.tt && sh.block == 512 && Mh.jz22 == 8 && Mh.jzm == 8) {
        switch (sh.spt) {
            case 2: return launch_mp_g<2, 512, 8, 8, true>(Mh, M, A, grid, st, occ);
            case 3: return launch_mp_g<3, 512, 8, 8, true>(Mh, M, A, grid, st, occ);
            case 4: return launch_mp_g<4, 512, 8, 8, true>(Mh, M, A, grid, st, occ);
            default: break;
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace csl
