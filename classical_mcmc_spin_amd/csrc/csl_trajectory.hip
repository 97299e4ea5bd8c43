// csl_trajectory.hip — the persistent batched RK4 kernel of atom-major
// launch shapes (kVariantAtomMajor): translation-invariant bond matrices and
// fields, no onsite matrix, the same number of bonds at every site.
//
// Compiled once per sites-per-thread value (CSL_SPT, set by the build); each
// object defines launch_trajectory_spt<CSL_SPT>.
//
// One workgroup per trajectory (or per piece of the work split, see
// PersistArgs); wave w owns units [start, start + units) of 64 cells of one
// sublattice (atom_major_tile), a lane one site of each unit.  A thread keeps
// the RK4 state x, the accumulator and the stage input of its own sites in
// VGPRs; the stage inputs of all sites live in two LDS buffers, so a stage is
// one gather, the field, the update, one store and one barrier.
//
// Everything that is not one of those four things is taken out of the stage:
//   * the field's constant part -(B + drive) of the stage times comes
//     from a small LDS table (one row per sublattice), written one step
//     ahead by the first waves; the pulse envelopes themselves are evaluated
//     for a chunk of steps at once, one lane per (step, stage time, pulse);
//   * a recorded step leaves four sums per wave (S and S.H); the rotation
//     into the sublattice frames, the staggered sign and the energy's B term
//     act on those sums, for a chunk of records at once and one wave per
//     record.
#include "csl_device.hpp"
#include "csl_record.hpp"

#ifndef CSL_SPT
#error "CSL_SPT (sites per thread) must be defined by the build"
#endif

namespace csl {

namespace {

// The kernel's argument block, read back from the kernel argument segment
// where it is used: the compiler cannot carry the scalars of rarely taken
// paths (records, seams) through the time loop in SGPRs.
struct TrajKernArgs {
    LatDev L;
    PersistArgs A;
    int chunk;
};
using KP = const TrajKernArgs __attribute__((address_space(4)))*;
__device__ __forceinline__ KP kern_args() {
    auto p = (unsigned long long)(__builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(p));
    return (KP)p;
}

// The waves that own NU units.  The barriers of a workgroup's waves pair up
// by count, whichever instance a wave runs.
template <int SPT, int NU, int ZMAX, bool DAMP, bool SAMP>
__device__ __forceinline__ void run_wave(const TrajKernArgs& K, double* smem, int wave, int wstart) {
    const int NP = K.L.NP, n_atoms = K.L.n_atoms, npad = K.L.npad;
    const int T = blockDim.x;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int nwaves = T >> 6;
    const int wpa = nwaves / n_atoms;
    const int atom = wave / wpa;
    const int C = K.chunk;
    // LDS: the stage inputs, both buffers of a site in one 48-byte record
    // [x y | x' y' | z z'] (a gather of either is one address and two
    // immediate offsets; separate planes, without the two-way bank conflicts
    // of z, cost as much in address arithmetic: 11.9 against 12.1 us a step
    // at 36x36), then the small tables
    double* const coef = smem + 6 * NP;          // [n_atoms][10][4] record weights of a wave's sums
    double* const cst = coef + 40 * n_atoms;     // [n_atoms][3][3]: B, d0, d1 of each component
    double* const hin = cst + 9 * n_atoms;       // [2 step parity][4][n_atoms][3]: the drive at the step's start,
                                                 // -(B + drive) at its middle and end, -B
    double* const drv = hin + 24 * n_atoms;      // [2 chunk parity][C][6] pulse envelopes
    double* const red = drv + 12 * C;            // [C][nwaves][4] record sums of the waves
    auto lds_ld = [&](int which, int q, double S[3]) {
        const double* r = smem + 6 * q;
        const double2 v = *reinterpret_cast<const double2*>(r + 2 * which);
        S[0] = v.x;
        S[1] = v.y;
        S[2] = r[4 + which];
    };
    auto lds_st = [&](int which, int q, const double S[3]) {
        double* r = smem + 6 * q;
        *reinterpret_cast<double2*>(r + 2 * which) = make_double2(S[0], S[1]);
        r[4 + which] = S[2];
    };

    const int pbase = atom * npad + wstart * kWave + lane;
    double x[NU][3], acc[NU][3], y[NU][3];
    // Twelve bonds and three sites a thread or more: partners two to a word,
    // and a stage's own value read back from LDS, or 470 bytes a lane spill
    // (600 trajectories of 36x36 x 200 steps: 11.3 -> 8.3 ms a call; at two
    // sites and fewer unpacking costs 7 %).
    constexpr bool kPack = ZMAX > 6 && SPT > 2;
    constexpr int kWords = kPack ? (ZMAX + 1) / 2 : ZMAX;
    int nb[NU][kWords];
#pragma unroll
    for (int m = 0; m < NU; ++m) {
        // padding lanes (no cell) hold a zero spin and gather themselves:
        // their field is finite and their derivative zero
        const int p = pbase + m * kWave;
        const bool real = p - atom * npad < K.L.n_cells;
#pragma unroll
        for (int k = 0; k < ZMAX; ++k) {
            const int q = real ? K.L.col[size_t(k) * NP + p] : p;
            if constexpr (!kPack) nb[m][k] = q;
            else nb[m][k >> 1] = k & 1 ? nb[m][k >> 1] | q << 16 : q;
        }
    }
    auto nbr = [&](int m, int k) {
        if constexpr (kPack) return int((unsigned(fresh(nb[m][k >> 1])) >> (16 * (k & 1))) & 0xffffu);
        else return nb[m][k];
    };
    const double dt = K.A.dt;
    const double b16 = (1.0 / 6.0) * dt, b13 = (1.0 / 3.0) * dt, hdt = 0.5 * dt;

    const int n_pieces = K.A.sched ? K.A.max_pieces : 1;
    for (int piece = 0; piece < n_pieces; ++piece) {
        int b = blockIdx.x, s_begin = 0, s_end = K.A.n_steps, slot_in = -1, slot_out = -1;
        if (K.A.sched) {
            const int* r = K.A.sched + (size_t(blockIdx.x) * K.A.max_pieces + piece) * 5;
            b = uniform(r[0]);
            s_begin = uniform(r[1]);
            s_end = uniform(r[2]);
            slot_in = uniform(r[3]);
            slot_out = uniform(r[4]);
            if (b < 0) continue;  // uniform
        }
        const bool drive_on = K.A.amp[2 * b] != 0.0 || K.A.amp[2 * b + 1] != 0.0;
        __syncthreads();  // the previous piece is done with the LDS
        if (slot_in < 0) {
            // initial state -> LDS (device order)
            const double* init = K.A.init + size_t(b) * K.A.init_stride;
            for (int p = tid; p < NP; p += T) {
                const int a = p / npad, cell = p - a * npad;
                double v[3] = {0.0, 0.0, 0.0};
                if (cell < K.L.n_cells) {
                    const size_t i = size_t(cell) * n_atoms + a;
                    v[0] = init[3 * i];
                    v[1] = init[3 * i + 1];
                    v[2] = init[3 * i + 2];
                }
                lds_st(0, p, v);
            }
        } else {
            // the state at step s_begin, saved by the workgroup that ran the
            // trajectory's first steps (it does so before anything else, so
            // the wait is short); a bounded wait that gives up flags the launch
            if (tid == 0) {
                unsigned ok = 0;
                for (long it = 0; it < (1L << 24); ++it) {
                    ok = __hip_atomic_load(K.A.flags + slot_in, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
                    if (ok) break;
                    __builtin_amdgcn_s_sleep(8);
                }
                if (!ok) __hip_atomic_store(K.A.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            __atomic_thread_fence(__ATOMIC_ACQUIRE);
            const double* sv = K.A.saved + size_t(slot_in) * 3 * size_t(NP);
            for (int p = tid; p < NP; p += T) {
                const double v[3] = {sv[3 * p], sv[3 * p + 1], sv[3 * p + 2]};
                lds_st(0, p, v);
            }
        }
        // small tables of this trajectory's Hamiltonian
        const double* mats = K.L.mats + size_t(b) * K.A.mats_stride;
        const double* field = K.L.field + size_t(b) * K.A.field_stride;
        for (int i = tid; i < 3 * n_atoms; i += T) {
            cst[3 * i] = field[i];
            cst[3 * i + 1] = K.L.fdrive[i];
            cst[3 * i + 2] = K.L.fdrive[3 * n_atoms + i];
            for (int par = 0; par < 2; ++par)  // without a drive the rows stay 0 and -B
                for (int st = 0; st < 4; ++st) hin[(par * 4 + st) * 3 * n_atoms + i] = st ? -field[i] : 0.0;
        }
        for (int i = tid; i < 40 * n_atoms; i += T) {
            // out[j] = sum over waves of coef[atom][j] . (Sx, Sy, Sz, e):
            // staggered, local and global magnetisation, energy: e = S.H with
            // the undriven H = -B + sum J S, so 1/2 (e - B.S)
            const int a = i / 40, j = (i / 4) % 10, e = i & 3;
            const int d = j % 3;
            double v = 0.0;
            if (e < 3 && j < 9) {
                v = j < 3 ? K.L.afm[a] * K.L.frames[a * 9 + d * 3 + e]
                          : (j < 6 ? (d == e ? 1.0 : 0.0) : K.L.frames[a * 9 + d * 3 + e]);
            } else if (j == 9) {
                v = e == 3 ? 0.5 : -0.5 * field[3 * a + e];
            }
            coef[i] = v;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < NU; ++m) lds_ld(0, pbase + m * kWave, x[m]);

        // Envelopes of steps n0 .. n0 + C - 1 into chunk buffer cp: lane =
        // (step, stage time, pulse); evaluated by the last wave, which owns
        // the fewest real sites (padding sits at the end).
        auto write_drive = [&](int n0, int cp) {
            if (drive_on && wave == nwaves - 1 && lane < 6 * C) {
                const KP G = kern_args();
                const int q = lane / 6, st = (lane % 6) >> 1, pl = lane & 1;
                const int n = n0 + q;
                if (n < s_end) {
                    const double t = G->A.tgrid[n];
                    const double ts = st == 0 ? t : (st == 1 ? t + 0.5 * dt : t + 1.0 * dt);
                    drv[cp * 6 * C + lane] =
                        drive_factor(G->A.amp[2 * b + pl], ts, G->A.t_pulse[2 * b + pl], G->L.width, G->L.freq);
                }
            }
        };
        // hin rows of the step whose envelopes are drv[f .. f+5]
        auto write_hin = [&](const double* f, int par) {
            if (drive_on && tid < 9 * n_atoms) {
                const int st = tid / (3 * n_atoms), i = tid - st * 3 * n_atoms;
                const double B = cst[3 * i], d0 = cst[3 * i + 1], d1 = cst[3 * i + 2];
                const double D = d0 * f[2 * st] + d1 * f[2 * st + 1];
                hin[par * 12 * n_atoms + tid] = st ? -B - D : D;
            }
        };
        write_drive(s_begin, 0);
        lds_barrier();
        write_hin(drv, 0);
        lds_barrier();

        // four sums of the wave (S and e) into red[slot][wave]
        auto reduce_obs = [&](int slot, const double s[3], double e) {
            wave_sum4(s[0], s[1], s[2], e, lane, red + (slot * nwaves + wave) * 4);
        };
        // records ri0 .. ri0 + cnt - 1 from red[0 .. cnt-1], one wave each
        auto publish = [&](int ri0, int cnt) {
            const KP G = kern_args();
            const double inv_n = 1.0 / double(G->L.N);
            for (int k = wave; k < cnt; k += nwaves) {
                if (lane < 10) {
                    double v = 0.0;
                    for (int w = 0; w < nwaves; ++w) {
                        const double* r = red + (k * nwaves + w) * 4;
                        const double* c = coef + ((w / wpa) * 10 + lane) * 4;
                        v += c[0] * r[0] + c[1] * r[1] + c[2] * r[2] + c[3] * r[3];
                    }
                    const size_t ri = size_t(ri0 + k);
                    if (lane < 9) {
                        if (G->A.mags) G->A.mags[(ri * G->A.B + b) * 9 + lane] = v * inv_n;
                    } else if (G->A.energy) {
                        G->A.energy[ri * G->A.B + b] = v * inv_n;
                    }
                }
            }
        };

        // Threads with few sites and three bonds keep their matrices in
        // registers and gather one bond ahead of the products: with two or
        // three waves per SIMD the scalar loads and the LDS latency show
        // (us a step, off -> on: 6x6 1.45 -> 1.26, 24x24 3.24 -> 3.07, 25
        // trajectories of 15x13 1.97 -> 1.81).  With three sites a thread and
        // more the registers run out (36x36: 11.9 -> 13.3), with six bonds
        // the matrices do (pyrochlore 4^3: 3.98 -> 4.45).
        constexpr bool kAhead = SPT <= 2 && ZMAX == 3;
        double Jh[kAhead ? 9 * ZMAX : 1];
        if constexpr (kAhead) {
#pragma unroll
            for (int q = 0; q < 9 * ZMAX; ++q) Jh[q] = (as_const(mats) + atom * ZMAX * 9)[q];
        }
        // One RK4 stage (compile-time index).  slot >= 0 in stage 0 of a
        // recorded step: the sums of the state go to red[slot].
        auto stage = [&](auto s_, int par, int slot) {
            constexpr int s = decltype(s_)::value;
            constexpr int cur = s & 1, nxt = 1 - (s & 1);
            constexpr int st = s == 0 ? 3 : (s == 3 ? 2 : 1);
            const double cdt = (s == 2) ? dt : hdt;
            const double bdt = (s == 0 || s == 3) ? b16 : b13;
            const double* h0 = hin + ((par * 4 + st) * n_atoms + atom) * 3;
            double H[NU][3];
            const double hx = h0[0], hy = h0[1], hz = h0[2];
            // the drive of stage 0, read before the bonds where registers
            // allow (24x24 2.5 % slower otherwise; 36x36 1.5 % with it)
            double D[3] = {0.0, 0.0, 0.0};
            auto load_drive = [&] {
#pragma unroll
                for (int d = 0; d < 3; ++d) D[d] = hin[(par * 4 * n_atoms + atom) * 3 + d];
            };
            if constexpr (s == 0 && kAhead) load_drive();
#pragma unroll
            for (int m = 0; m < NU; ++m) {
                H[m][0] = hx;
                H[m][1] = hy;
                H[m][2] = hz;
            }
            // bond by bond, one FMA chain per field component
            if constexpr (kAhead) {
#pragma unroll
                for (int q = 0; q < 9 * ZMAX; ++q) {
                    // the same matrices, kept where they are
                    if constexpr (SPT == 1) asm volatile("" : "+v"(Jh[q]));
                    else asm volatile("" : "+s"(Jh[q]));
                }
                double S[NU][3];
#pragma unroll
                for (int m = 0; m < NU; ++m) lds_ld(cur, nbr(m, 0), S[m]);
#pragma unroll
                for (int k = 0; k < ZMAX; ++k) {
#pragma unroll
                    for (int m = 0; m < NU; ++m) {
#pragma unroll
                        for (int e = 0; e < 3; ++e)
#pragma unroll
                            for (int d = 0; d < 3; ++d) H[m][d] = fma(Jh[k * 9 + d * 3 + e], S[m][e], H[m][d]);
                        if (k + 1 < ZMAX) lds_ld(cur, nbr(m, k + 1), S[m]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            } else {
                // one bond matrix (scalar loads, shared by the wave's sites)
                // live at a time
                cptr<double> Jt = as_const(mats) + atom * ZMAX * 9 + opaque_zero();
#pragma unroll
                for (int k = 0; k < ZMAX; ++k) {
                    double J[9];
#pragma unroll
                    for (int q = 0; q < 9; ++q) J[q] = Jt[k * 9 + q];
#pragma unroll
                    for (int m = 0; m < NU; ++m) {
                        double S[3];
                        lds_ld(cur, nbr(m, k), S);
#pragma unroll
                        for (int e = 0; e < 3; ++e)
#pragma unroll
                            for (int d = 0; d < 3; ++d) H[m][d] = fma(J[d * 3 + e], S[e], H[m][d]);
                    }
                }
            }
            // damped: a unit's root and division make a branch, into which the
            // compiler puts off the field's products and the updates of the
            // other units with all their operands: 300 to 2600 bytes a lane of
            // spills, and 24x24 with twelve bonds 64 x 200 steps 4.3 ms
            // against 2.0 with the field and each unit's update held
            if constexpr (DAMP) {
#pragma unroll
                for (int m = 0; m < NU; ++m) hold(H[m]);
            }
            if (s == 0 && slot >= 0) {
                double sm[3] = {0.0, 0.0, 0.0}, e = 0.0;
#pragma unroll
                for (int m = 0; m < NU; ++m) {
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        sm[d] += x[m][d];
                        e = fma(x[m][d], H[m][d], e);
                    }
                }
                reduce_obs(slot, sm, e);
            }
            if constexpr (s == 0) {
                // the record's energy is the undriven field's: the drive comes
                // after it (a driven field would round at the drive's size)
                if constexpr (!kAhead) load_drive();
#pragma unroll
                for (int m = 0; m < NU; ++m)
#pragma unroll
                    for (int d = 0; d < 3; ++d) H[m][d] -= D[d];
            }
#pragma unroll
            for (int m = 0; m < NU; ++m) {
                double own[3];
                if constexpr (kPack && s > 0) lds_ld(cur, fresh(pbase + m * kWave), own);
                const double* Sm = s == 0 ? x[m] : (kPack ? own : y[m]);
                double k[3];
                if constexpr (DAMP) {
                    ll_su2_guarded(H[m], Sm, K.L.alpha, k);
                } else {
                    k[0] = H[m][1] * Sm[2] - H[m][2] * Sm[1];
                    k[1] = H[m][2] * Sm[0] - H[m][0] * Sm[2];
                    k[2] = H[m][0] * Sm[1] - H[m][1] * Sm[0];
                }
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    if (s == 0) acc[m][d] = x[m][d] + bdt * k[d];
                    else if (s < 3) acc[m][d] = acc[m][d] + bdt * k[d];
                    else x[m][d] = acc[m][d] + bdt * k[d];
                    if (s < 3) y[m][d] = x[m][d] + cdt * k[d];
                }
                if constexpr (DAMP) {
                    if constexpr (s < 3) {
                        hold(acc[m]);
                        hold(y[m]);
                    } else {
                        hold(x[m]);
                    }
                }
                lds_st(nxt, pbase + m * kWave, s < 3 ? y[m] : x[m]);
            }
            lds_barrier();
        };

        // time loop in chunks of C steps; the next record index and the step
        // it belongs to advance by counters
        const int si = K.A.save_interval;
        int ri = (s_begin + si - 1) / si;      // first record at or after s_begin
        int next_rec = ri * si;
        int smp = 0, next_smp = -1;            // next state sample
        if constexpr (SAMP) {
            const int se = K.A.sample_every;
            smp = (s_begin + se - 1) / se;
            next_smp = smp < K.A.n_samples ? smp * se : -1;
        }
        for (int n0 = s_begin, cp = 0; n0 < s_end; n0 += C, cp ^= 1) {
            const int n1 = min(n0 + C, s_end);
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
                if (SAMP && n == next_smp) {
                    const KP G = kern_args();
                    double* row = sample_row(G->A.samples, G->A.B, n_atoms, G->L.n_cells, smp, b, atom);
#pragma unroll
                    for (int m = 0; m < NU; ++m) {
                        const int cell = pbase + m * kWave - atom * npad;
                        if (cell < G->L.n_cells) {
#pragma unroll
                            for (int d = 0; d < 3; ++d) row[size_t(d) * G->L.n_cells + cell] = x[m][d];
                        }
                    }
                    ++smp;
                    next_smp = smp < G->A.n_samples ? next_smp + G->A.sample_every : -1;
                }
                const int q = n + 1 - n0;
                if (n + 1 < s_end && q < C) write_hin(drv + (cp * C + q) * 6, par ^ 1);
                stage(std::integral_constant<int, 0>{}, par, slot);
                if (n + 1 == n1 && ri > ri0) publish(ri0, ri - ri0);
                stage(std::integral_constant<int, 1>{}, par, -1);
                // the next chunk's envelopes are complete since stage 0
                if (n + 1 < s_end && q == C) write_hin(drv + (cp ^ 1) * C * 6, par ^ 1);
                stage(std::integral_constant<int, 2>{}, par, -1);
                stage(std::integral_constant<int, 3>{}, par, -1);
            }
        }

        const KP G = kern_args();
        if (slot_out >= 0) {
            // hand the state at s_end to the piece that continues the trajectory
            double* sv = G->A.saved + size_t(slot_out) * 3 * size_t(NP);
#pragma unroll
            for (int m = 0; m < NU; ++m) {
                const int p = pbase + m * kWave;
#pragma unroll
                for (int d = 0; d < 3; ++d) sv[3 * p + d] = x[m][d];
            }
            __threadfence();
            __syncthreads();
            if (tid == 0) __hip_atomic_store(G->A.flags + slot_out, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        // final record: state after the last step (lattice_gpu.cu:567-568)
        if (s_end == G->A.n_steps) {
            double sm[3] = {0.0, 0.0, 0.0}, e = 0.0;
#pragma unroll
            for (int m = 0; m < NU; ++m) {
                double H[3] = {-field[atom * 3], -field[atom * 3 + 1], -field[atom * 3 + 2]};
#pragma unroll
                for (int k = 0; k < ZMAX; ++k) {
                    double S[3];
                    lds_ld(0, nbr(m, k), S);
                    add_bond_fused(as_const(mats) + (atom * ZMAX + k) * 9, S, H);
                }
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    sm[d] += x[m][d];
                    e = fma(x[m][d], H[d], e);
                }
            }
            reduce_obs(0, sm, e);
            lds_barrier();
            publish(G->A.n_rec - 1, 1);
            if (G->A.final_states) {
                double* out = G->A.final_states + size_t(b) * G->L.N * 3;
#pragma unroll
                for (int m = 0; m < NU; ++m) {
                    const int cell = pbase + m * kWave - atom * npad;
                    if (cell < G->L.n_cells) {
                        const size_t i = size_t(cell) * n_atoms + atom;
                        out[3 * i] = x[m][0];
                        out[3 * i + 1] = x[m][1];
                        out[3 * i + 2] = x[m][2];
                    }
                }
            }
        }
    }  // pieces
}

}  // namespace

// SPT: the most units a wave owns; the others own one less.  SAMP: the launch
// stores state samples (without them the test alone costs 3 % at 24x24).
template <int SPT, int ZMAX, bool DAMP, bool SAMP>
__global__ void __launch_bounds__(persistent_max_block<SPT>()) k_trajectory(TrajKernArgs K) {
    extern __shared__ double smem[];
    const int wave = uniform(threadIdx.x >> 6);
    int wstart = 0, wunits = 0;
    atom_major_tile(blockDim.x >> 6, K.L.n_atoms, K.L.npad / kWave, wave, wstart, wunits);
    wstart = uniform(wstart);
    wunits = uniform(wunits);
    if (SPT == 1 || wunits == SPT) run_wave<SPT, SPT, ZMAX, DAMP, SAMP>(K, smem, wave, wstart);
    else run_wave<SPT, (SPT > 1 ? SPT - 1 : 1), ZMAX, DAMP, SAMP>(K, smem, wave, wstart);
}

namespace {

template <int SPT, int ZMAX, bool DAMP, bool SAMP>
hipError_t launch_t(const TrajKernArgs& K, int block, size_t lds, hipStream_t st, int* occ) {
    auto kern = k_trajectory<SPT, ZMAX, DAMP, SAMP>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, kern, block, lds);
    hipLaunchKernelGGL(kern, dim3(K.A.sched ? K.A.grid : K.A.B), dim3(block), lds, st, K);
    return hipGetLastError();
}

template <int SPT, int ZMAX>
hipError_t launch_t_damp(const TrajKernArgs& K, int block, size_t lds, hipStream_t st, int* occ) {
    const bool damp = K.L.alpha > 0.0, samp = K.A.sample_every > 0;
    if (samp)
        return damp ? launch_t<SPT, ZMAX, true, true>(K, block, lds, st, occ)
                    : launch_t<SPT, ZMAX, false, true>(K, block, lds, st, occ);
    return damp ? launch_t<SPT, ZMAX, true, false>(K, block, lds, st, occ)
                : launch_t<SPT, ZMAX, false, false>(K, block, lds, st, occ);
}

}  // namespace

template <>
hipError_t launch_trajectory_spt<CSL_SPT>(const LatDev& L, const PersistArgs& A, int block, hipStream_t st, int* occ) {
    const int chunk = trajectory_chunk(L, block);
    if (!chunk) return hipErrorInvalidValue;
    const TrajKernArgs K{L, A, chunk};
    const size_t lds = trajectory_lds_bytes(L, block, chunk);
    switch (L.zmax) {
        case 3: return launch_t_damp<CSL_SPT, 3>(K, block, lds, st, occ);
        case 6: return launch_t_damp<CSL_SPT, 6>(K, block, lds, st, occ);
        case 12: return launch_t_damp<CSL_SPT, 12>(K, block, lds, st, occ);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace csl
