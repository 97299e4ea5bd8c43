// csl_adjoint_sweep.hip — backward sweep of the discrete adjoint with the
// parameter terms summed on the way (formulas in csl_adjoint.hip), for
// lattices with three bonds at every site, per-sublattice fields and no
// onsite matrix.
//
// The parameter terms are u_i . (sum_k dJ_kp S_p(k) - dB_p) over all sites,
// stages and steps, and dJ, dB are constants of the sublattice: with
//   G_ak = sum u_i (x) S_p(k)   (3x3, sites of sublattice a),   U_a = sum u_i
// the gradient is sum_ak dJ_pak : G_ak - sum_a dB_pa . U_a.  The sweep has
// u_i in registers and gathers every S_p(k) for the field anyway, so a site's
// terms are 30 FMAs of registers instead of a 24-byte store of u_i, its
// reload and the partners' by another kernel, and 150 FMAs there (five
// parameters).  The cotangents never leave the chip, and the memory of a run
// halves.  32 starts of the 24x24 lattice x 2000 steps: 20.4 ms here, against
// 24 ms of k_adj_bwd and 18 ms of k_adj_par, which ran beside it only while
// its stream had a hardware queue of its own (a gradient 32.5 ms, before 37
// or, with other handles alive, 53); 4 starts of 12x12 x 250 steps 1.15 ms.
//
// A wave owns units of 64 cells of one sublattice (atom_major_tile), so all
// its sites share one set of sums and bond matrices.  One barrier a stage
// slot, with two y and two u buffers in LDS as in k_adj_bwd
// (csl_adjoint.hip).  What a step needs besides its states (fields at the
// three stage times, the loss cotangent) comes ready from k_adj_rows as three
// uniform values a slot: computed here, they held enough scalars and lanes to
// push the prefetched states to scratch, and a slot waited for them to come
// from memory (30.6 ms).  A site without a spin (padding) is no branch: one a
// unit kept the units' gathers from overlapping (23.7 ms).
//
// Rounding: a thread sums at most 16 steps of its own sites, the wave's sums
// of those blocks go to running totals at the steps' multiples of 16 whatever
// the segments, so every checkpoint spacing gives the same bits.
//
// What bounds it: FP64 issue on the busiest SIMD, which carries 5 of the 18
// units of 24x24 (1000 VALU instructions a slot on two waves, 1.8 of the
// 2.5 us); B starts use B CUs.
#include <algorithm>

#include "csl_device.hpp"
#include "csl_record.hpp"

namespace csl {

namespace {

constexpr int kZ = 3;            // bonds per site
constexpr int kSums = 9 * kZ + 3;  // sums per thread: G_k, U
constexpr int kRow = 12;           // doubles per (trajectory, step, sublattice): see k_adj_rows

constexpr int kMaxBlock = 512;     // two waves per SIMD with 256 VGPRs each (four units spill a little)

// The kernel's argument block, read back from the kernel argument segment by
// the code outside the loops, so that the loops do not carry it in SGPRs
// (the bond matrices of a sublattice take 54 of the 102).
struct SweepArgs {
    LatDev L;
    AdjArgs A;
};
using KP = const SweepArgs __attribute__((address_space(4)))*;
__device__ __forceinline__ KP kern_args() {
    auto p = (unsigned long long)(__builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(p));
    return (KP)p;
}

__device__ __forceinline__ void cross3(const double a[3], const double b[3], double o[3]) {
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}

// LDS: both y buffers of a site in one 48-byte record [x y | x' y' | z z'],
// then the same for u
struct Lds2 {
    double* a;
    __device__ __forceinline__ void load(int which, int q, double S[3]) const {
        const double* r = a + 6 * q;
        const double2 v = *reinterpret_cast<const double2*>(r + 2 * which);
        S[0] = v.x;
        S[1] = v.y;
        S[2] = r[4 + which];
    }
    __device__ __forceinline__ void store(int which, int q, const double S[3]) const {
        double* r = a + 6 * q;
        *reinterpret_cast<double2*>(r + 2 * which) = make_double2(S[0], S[1]);
        r[4 + which] = S[2];
    }
};

template <int NU, bool DAMP>
__device__ __forceinline__ void sweep_wave(double* smem, int wave, int wstart) {
    const KP K = kern_args();
    const int NP = K->L.NP, n_atoms = K->L.n_atoms, npad = K->L.npad;
    const int b = blockIdx.x, T = blockDim.x, tid = threadIdx.x;
    const int lane = tid & (kWave - 1), nwaves = T >> 6;
    const int atom = wave / (nwaves / n_atoms);
    const Lds2 Yl{smem}, Ul{smem + 6 * NP};
    double* const sums = smem + 12 * NP;   // [nwaves][32]
    const double dt = K->A.dt, alpha = DAMP ? K->L.alpha : 0.0;
    const double b16 = (1.0 / 6.0) * dt, b13 = (1.0 / 3.0) * dt, hdt = 0.5 * dt;
    const size_t SZ = size_t(3) * NP;
    const double* const mats = K->L.mats + size_t(b) * K->A.mats_stride + atom * kZ * 9;
    const int n0 = K->A.n0, n1 = K->A.n1;  // stage slots q = 4 n + s of these steps
    const double* const Yb = K->A.Y + (size_t(b) * K->A.seg_len - K->A.y0) * 4 * SZ;
    const double* const rows = K->A.rows + (size_t(b) * (K->A.seg_len + 1) * n_atoms + atom) * kRow;

    const int pbase = atom * npad + wstart * kWave + lane;
    int nb[NU][kZ];
    // padding lanes (of a sublattice's last unit) hold zeros and gather themselves
    const bool last_real = pbase + (NU - 1) * kWave - atom * npad < int(K->L.n_cells);
#pragma unroll
    for (int m = 0; m < NU; ++m) {
        const int p = pbase + m * kWave;
#pragma unroll
        for (int k = 0; k < kZ; ++k) nb[m][k] = m < NU - 1 || last_real ? K->L.col[size_t(k) * NP + p] : p;
    }

    double lam[NU][3], acc[NU][3], c[NU][3], dir[NU][3], pre[NU][3];
    double G[kZ][9], U[3], run = 0.0;  // run: lane k's running total of the wave's sum k

    // row of step n and this sublattice (k_adj_rows)
    auto row = [&](int n) { return as_const(rows) + size_t(n) * n_atoms * kRow; };
    // -(B + drive) of stage slot q
    auto load_h = [&](int q, double h[3]) __attribute__((always_inline)) {
        cptr<double> r = row(q >> 2) + 3 * (((q & 3) + 1) >> 1);  // t, t + dt/2, t + dt/2, t + dt
#pragma unroll
        for (int d = 0; d < 3; ++d) h[d] = r[d];
    };
    auto fetch = [&](int q) __attribute__((always_inline)) {
        const double* src = Yb + size_t(q) * SZ;
#pragma unroll
        for (int m = 0; m < NU; ++m) {
            const int p = fresh(pbase + m * kWave);
            const double2 v = reinterpret_cast<const double2*>(src)[p];
            pre[m][0] = v.x;
            pre[m][1] = v.y;
            pre[m][2] = src[2 * NP + p];
        }
    };
    auto put = [&](int yi) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NU; ++m) Yl.store(yi, fresh(pbase + m * kWave), pre[m]);
    };
    // the thread sums -> the wave's running totals
    auto flush = [&]() __attribute__((always_inline)) {
        double* r = sums + wave * 32;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            double v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                constexpr int kG = 9 * kZ;
                const int k = 4 * i + j;
                v[j] = k < kG ? G[k < kG ? k / 9 : 0][k % 9] : (k < kSums ? U[k >= kG && k < kSums ? k - kG : 0] : 0.0);
            }
            wave_sum4(v[0], v[1], v[2], v[3], lane, r + 4 * i);
        }
        run += r[lane & 31];
    };
    // the bond matrices of the sublattice, read once a slot (kept over the
    // loop they would push other scalars out of the SGPRs)
    auto load_j = [&](double (&J)[kZ][9]) __attribute__((always_inline)) {
        cptr<double> src = as_const(mats) + opaque_zero();
#pragma unroll
        for (int k = 0; k < kZ; ++k)
#pragma unroll
            for (int j = 0; j < 9; ++j) J[k][j] = src[k * 9 + j];
    };
    // A: u -> LDS and the sums, the field at the state in y buffer PAR, the
    // direct term -> dir
    auto vjp_a = [&](auto par_, const double h0[3], const double (&J)[kZ][9]) __attribute__((always_inline)) {
        constexpr int PAR = decltype(par_)::value;
        // u = S x w needs no field
#pragma unroll
        for (int m = 0; m < NU; ++m) {
            const int p = fresh(pbase + m * kWave);
            const double* v = c[m];
            double S[3], u[3], H[3];
            Yl.load(PAR, p, S);
            double inv = 0.0, w[3];
            if constexpr (DAMP) {
                const double n2 = S[0] * S[0] + S[1] * S[1] + S[2] * S[2];
                inv = rsqrt_nr(n2 > 0.0 ? n2 : 1.0);  // 0 (padding): every term below is 0
                double vxS[3];
                cross3(v, S, vxS);
#pragma unroll
                for (int d = 0; d < 3; ++d) w[d] = v[d] - alpha * inv * vxS[d];
            } else {
#pragma unroll
                for (int d = 0; d < 3; ++d) w[d] = v[d];
            }
            cross3(S, w, u);
            Ul.store(PAR, p, u);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                U[d] += u[d];
                H[d] = h0[d];
            }
#pragma unroll
            for (int k = 0; k < kZ; ++k) {
                double s[3];
                Yl.load(PAR, fresh(nb[m][k]), s);
#pragma unroll
                for (int e = 0; e < 3; ++e)
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        H[d] = fma(J[k][d * 3 + e], s[e], H[d]);
                        G[k][d * 3 + e] = fma(u[d], s[e], G[k][d * 3 + e]);
                    }
                hold(H);
                hold(G[k]);
            }
            if constexpr (DAMP) {
                double cc[3], cxv[3], Sxc[3], wxH[3];
                cross3(H, S, cc);
                cross3(cc, v, cxv);
                cross3(S, cc, Sxc);
                cross3(w, H, wxH);
                const double k3 = alpha * inv * inv * inv * (v[0] * Sxc[0] + v[1] * Sxc[1] + v[2] * Sxc[2]);
#pragma unroll
                for (int d = 0; d < 3; ++d) dir[m][d] = wxH[d] - alpha * inv * cxv[d] + k3 * S[d];
            } else {
                cross3(v, H, dir[m]);
            }
        }
    };
    // B: mu = direct + sum_k J_k u_p(k) of the stage above (u buffer PAR),
    // then the cotangent c = w_lam lambda + w_mu mu of the next
    auto vjp_b = [&](auto par_, const double (&J)[kZ][9]) __attribute__((always_inline)) {
        constexpr int PAR = decltype(par_)::value;
#pragma unroll
        for (int k = 0; k < kZ; ++k) {
#pragma unroll
            for (int m = 0; m < NU; ++m) {
                double up[3];
                Ul.load(PAR, fresh(nb[m][k]), up);
#pragma unroll
                for (int e = 0; e < 3; ++e)
#pragma unroll
                    for (int d = 0; d < 3; ++d) dir[m][d] = fma(J[k][d * 3 + e], up[e], dir[m][d]);
                hold(dir[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < NU; ++m)
#pragma unroll
            for (int d = 0; d < 3; ++d) acc[m][d] += dir[m][d];
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;

    // B ends step n: lambda_n = lambda' + mu's + d l_n / d x_n (in the first
    // slot of a launch that continues a sweep they are in lambda already)
    auto end_step = [&](int n, bool dl) __attribute__((always_inline)) {
        cptr<double> r = row(n) + 9;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double v = dl ? r[d] : 0.0;
#pragma unroll
            for (int m = 0; m < NU; ++m) lam[m][d] = acc[m][d] + (m < NU - 1 || last_real ? v : 0.0);
        }
    };

    // lambda at the end of the segment; no cotangents above it
    const bool first = K->A.first;
    auto lam_slot = [&](int m, int d) {
        const KP P = kern_args();
        return P->A.lam + size_t(b) * SZ + size_t(d) * NP + pbase + m * kWave;
    };
    // a thread's sum k as handed between segments (kSums: the running total)
    auto sum_slot = [&](int k) { return kern_args()->A.part + (size_t(b) * (kSums + 1) + k) * T + tid; };
    const double zero[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < NU; ++m) {
        Ul.store(0, pbase + m * kWave, zero);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            acc[m][d] = first ? 0.0 : *lam_slot(m, d);
            dir[m][d] = 0.0;
        }
    }

    // Slot q (one barrier each): B of slot q + 1 and A of slot q, buffers by
    // the parity of q.  y of slot q - 1 is fetched at the start and stored
    // into the free LDS buffer at the end.  The thread sums of up to 16 steps
    // go to the running totals at the steps' multiples of 16, so that every
    // segment layout adds alike.
    fetch(4 * n1 - 1);
    put(1);
    __syncthreads();
    bool dl = first;
    int top = n1;
#pragma unroll 1
    while (top > n0) {
        const int lo = max(n0, (top - 1) & ~15);
        const bool carry = top == n1 && !first;
#pragma unroll
        for (int k = 0; k < kZ; ++k)
#pragma unroll
            for (int j = 0; j < 9; ++j) G[k][j] = carry ? *sum_slot(k * 9 + j) : 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) U[j] = carry ? *sum_slot(9 * kZ + j) : 0.0;
        if (carry) run = *sum_slot(kSums);
#pragma unroll 1
        for (int n = top - 1; n >= lo; --n) {
#pragma unroll 1
            for (int h = 1; h >= 0; --h) {
                {   // slot 4 n + 3 (h = 1: the step above is complete) or 4 n + 1
                    const int q = 4 * n + 2 * h + 1;
                    double J[kZ][9], h0[3];
                    load_j(J);
                    load_h(q, h0);
                    fetch(q - 1);
                    vjp_b(P0{}, J);
                    if (h) {
                        end_step(n + 1, dl);
                        dl = true;
#pragma unroll
                        for (int m = 0; m < NU; ++m)
#pragma unroll
                            for (int d = 0; d < 3; ++d) {
                                acc[m][d] = lam[m][d];
                                c[m][d] = b16 * lam[m][d];
                            }
                    } else {
#pragma unroll
                        for (int m = 0; m < NU; ++m)
#pragma unroll
                            for (int d = 0; d < 3; ++d) c[m][d] = b13 * lam[m][d] + hdt * dir[m][d];
                    }
                    vjp_a(P1{}, h0, J);
                    put(0);
                    lds_barrier();
                }
                {   // slot 4 n + 2 or 4 n
                    const int q = 4 * n + 2 * h;
                    double J[kZ][9], h0[3];
                    load_j(J);
                    load_h(q, h0);
                    fetch(max(q - 1, 4 * n0));
                    vjp_b(P1{}, J);
                    const double wl = h ? b13 : b16, wm = h ? dt : hdt;
#pragma unroll
                    for (int m = 0; m < NU; ++m)
#pragma unroll
                        for (int d = 0; d < 3; ++d) c[m][d] = wl * lam[m][d] + wm * dir[m][d];
                    vjp_a(P0{}, h0, J);
                    put(1);
                    lds_barrier();
                }
            }
        }
        if ((lo & 15) == 0) flush();
        top = lo;
    }
    {
        double J[kZ][9];
        load_j(J);
        vjp_b(P0{}, J);
        end_step(n0, true);
    }
    if (n0 > 0) {
        // hand lambda and the sums to the next (earlier) segment
#pragma unroll
        for (int m = 0; m < NU; ++m)
#pragma unroll
            for (int d = 0; d < 3; ++d) *lam_slot(m, d) = lam[m][d];
#pragma unroll
        for (int k = 0; k < kZ; ++k)
#pragma unroll
            for (int j = 0; j < 9; ++j) *sum_slot(k * 9 + j) = n0 & 15 ? G[k][j] : 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) *sum_slot(9 * kZ + j) = n0 & 15 ? U[j] : 0.0;
        *sum_slot(kSums) = run;
        return;
    }
    const KP E = kern_args();
    if (E->A.grad_init) {
        double* gi = E->A.grad_init + size_t(b) * E->L.N * 3;
#pragma unroll
        for (int m = 0; m < NU; ++m) {
            const int cell = pbase + m * kWave - atom * npad;
            if (m < NU - 1 || last_real) {
                const size_t i = size_t(cell) * n_atoms + atom;
                gi[3 * i] = lam[m][0];
                gi[3 * i + 1] = lam[m][1];
                gi[3 * i + 2] = lam[m][2];
            }
        }
    }
    // the waves' totals (flushed at step 0), then the parameters'
    // contractions, a thread each
    if (lane < 32) sums[wave * 32 + lane] = run;
    __syncthreads();
    if (tid < E->A.P) {
        const int wpa = nwaves / n_atoms;
        double g = 0.0;
        for (int a = 0; a < n_atoms; ++a) {
            const double* dJ = E->A.dmats + (size_t(tid) * n_atoms + a) * kZ * 9;
            const double* dB = E->A.dfield + (size_t(tid) * n_atoms + a) * 3;
            for (int k = 0; k < kSums; ++k) {
                double s = 0.0;
                for (int w = 0; w < wpa; ++w) s += sums[(a * wpa + w) * 32 + k];
                g += (k < 9 * kZ ? dJ[k] : -dB[k - 9 * kZ]) * s;
            }
        }
        E->A.grad[size_t(b) * E->A.P + tid] = g;
    }
}

}  // namespace

// What the sweep needs of a step of its segment besides the states, a thread
// per (trajectory, step, sublattice): -(B + drive) at the step's three stage times and
// d l_n / d x_n, so that the sequential sweep reads three uniform values a
// stage; and the loss term of the record.
__global__ void __launch_bounds__(256) k_adj_rows(LatDev L, AdjArgs A) {
    const size_t n_rec = size_t(A.n_steps) + 1, n_seg = size_t(A.n1 - A.n0) + 1, i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n_seg * A.B * L.n_atoms) return;
    const int atom = int(i % L.n_atoms);
    const size_t n = A.n0 + i / L.n_atoms % n_seg, b = i / L.n_atoms / n_seg;
    double* out = A.rows + ((b * (A.seg_len + 1) + n) * L.n_atoms + atom) * kRow;
    const double* B = L.field + b * A.field_stride + atom * 3;
    for (int sg = 0; sg < 3; ++sg) {
        double f[2] = {0.0, 0.0};
        if (A.fac && n < size_t(A.n_steps))
            for (int pl = 0; pl < 2; ++pl) f[pl] = A.fac[((n * 3 + sg) * A.B + b) * 2 + pl];
        for (int d = 0; d < 3; ++d)
            out[sg * 3 + d] =
                -B[d] - (L.fdrive[atom * 3 + d] * f[0] + L.fdrive[(L.n_atoms + atom) * 3 + d] * f[1]);
    }
    double dl[9], loss = 0.0;
    for (int j = 0; j < 9; ++j) {
        const double d = A.rec[(n * A.B + b) * 9 + j] - A.target[n * 9 + j];
        dl[j] = 2.0 * A.w[j] * d / double(L.N);
        loss += A.w[j] * d * d;
    }
    for (int e = 0; e < 3; ++e) {
        double v = dl[3 + e];
        for (int d = 0; d < 3; ++d) v += L.frames[atom * 9 + d * 3 + e] * (L.afm[atom] * dl[d] + dl[6 + d]);
        out[9 + e] = v;
    }
    if (atom == 0) A.loss_n[b * n_rec + n] = loss;
}

// SPT: the most units a wave owns; the others own one less.
template <int SPT, bool DAMP>
__global__ void __launch_bounds__(kMaxBlock) k_adj_sweep(SweepArgs K) {
    extern __shared__ double smem[];
    const int wave = uniform(threadIdx.x >> 6);
    int start = 0, units = 0;
    atom_major_tile(blockDim.x >> 6, K.L.n_atoms, K.L.npad / kWave, wave, start, units);
    start = uniform(start);
    units = uniform(units);
    if (SPT == 1 || units == SPT) sweep_wave<SPT, DAMP>(smem, wave, start);
    else sweep_wave<(SPT > 1 ? SPT - 1 : 1), DAMP>(smem, wave, start);
}

namespace {

struct SweepShape {
    int block, spt;
};

size_t sweep_lds(const LatDev& L, int block) {
    return sizeof(double) * (12 * size_t(L.NP) + size_t(block / kWave) * 32);
}

// The waves per sublattice whose busiest SIMD carries the fewest units (a
// slot ends when that SIMD is done); ties: the fewest units per wave.
// block 0: none.
SweepShape sweep_shape(const LatDev& L) {
    SweepShape best{0, 0};
    if (!(L.uniform && L.site_uniform && !L.has_onsite && L.full_coord && L.zmax == kZ)) return best;
    const int U = L.npad / kWave;
    int best_load = 1 << 30;
    for (int wpa = 1; wpa <= U; ++wpa) {
        const int spt = (U + wpa - 1) / wpa, block = L.n_atoms * wpa * kWave;
        if (spt > 4 || block > kMaxBlock || sweep_lds(L, block) > kLdsBytes) continue;
        const int load = atom_major_max_load(block / kWave, L.n_atoms, U);
        if (load < best_load || (load == best_load && spt < best.spt)) {
            best = {block, spt};
            best_load = load;
        }
    }
    return best;
}

template <int SPT, bool DAMP>
hipError_t launch_s(const LatDev& L, const AdjArgs& A, int block, hipStream_t st) {
    auto kern = k_adj_sweep<SPT, DAMP>;
    const size_t lds = sweep_lds(L, block);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(A.B), dim3(block), lds, st, SweepArgs{L, A});
    return hipGetLastError();
}

template <bool DAMP>
hipError_t launch_s_spt(const LatDev& L, const AdjArgs& A, const SweepShape& sh, hipStream_t st) {
    switch (sh.spt) {
        case 1: return launch_s<1, DAMP>(L, A, sh.block, st);
        case 2: return launch_s<2, DAMP>(L, A, sh.block, st);
        case 3: return launch_s<3, DAMP>(L, A, sh.block, st);
        case 4: return launch_s<4, DAMP>(L, A, sh.block, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool adjoint_sweep_fits(const LatDev& L) { return sweep_shape(L).block > 0; }

size_t adjoint_row_doubles(const LatDev& L) { return size_t(L.n_atoms) * kRow; }

hipError_t launch_adjoint_rows(const LatDev& L, const AdjArgs& A, hipStream_t st) {
    const size_t n = (size_t(A.n1 - A.n0) + 1) * A.B * L.n_atoms;
    hipLaunchKernelGGL(k_adj_rows, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, L, A);
    return hipGetLastError();
}

size_t adjoint_sweep_doubles(const LatDev& L) { return size_t(sweep_shape(L).block) * (kSums + 1); }

hipError_t launch_adjoint_sweep(const LatDev& L, const AdjArgs& A, hipStream_t st) {
    const SweepShape sh = sweep_shape(L);
    return L.alpha > 0.0 ? launch_s_spt<true>(L, A, sh, st) : launch_s_spt<false>(L, A, sh, st);
}

}  // namespace csl
