// csl_mixed_lds.hpp — LDS access, field rows, pulse envelopes and records
// shared by the persistent kernels of the mixed lattice (csl_mixed_waves.hip,
// csl_mixed_persist.hip).
#pragma once

#include "csl_mixed_device.hpp"
#include "csl_record.hpp"

namespace csl {

namespace {

// Kernel arguments, read back from the kernel argument segment where rarely
// taken paths need them (the compiler cannot carry them through the time
// loop in SGPRs).
struct MixKernArgs {
    const MixDev* M;
    MixPersistArgs A;
};
using MixArgsP = const MixKernArgs __attribute__((address_space(4)))*;
__device__ __forceinline__ MixArgsP mix_kern_args() {
    auto p = (unsigned long long)(__builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(p));
    return (MixArgsP)p;
}

__device__ __forceinline__ int lo16(unsigned v) { return int(v & 0xffffu); }
__device__ __forceinline__ int hi16(unsigned v) { return int(v >> 16); }
__device__ __forceinline__ void unpack8(const uint4& v, int q[8]) {
    q[0] = lo16(v.x); q[1] = hi16(v.x); q[2] = lo16(v.y); q[3] = hi16(v.y);
    q[4] = lo16(v.z); q[5] = hi16(v.z); q[6] = lo16(v.w); q[7] = hi16(v.w);
}

// 3-component value at r (8-byte aligned), 8-component value at (r6, r2)
__device__ __forceinline__ void ld3(const double* r, double v[3]) {
    v[0] = r[0];
    v[1] = r[1];
    v[2] = r[2];
}
__device__ __forceinline__ void ld8(const double* r6, const double* r2, double v[8]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double2 a = reinterpret_cast<const double2*>(r6)[i];
        v[2 * i] = a.x;
        v[2 * i + 1] = a.y;
    }
    const double2 a = *reinterpret_cast<const double2*>(r2);
    v[6] = a.x;
    v[7] = a.y;
}
__device__ __forceinline__ void st8(double* r6, double* r2, const double v[8]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) reinterpret_cast<double2*>(r6)[i] = make_double2(v[2 * i], v[2 * i + 1]);
    *reinterpret_cast<double2*>(r2) = make_double2(v[6], v[7]);
}

// Ends a bond: the field values as they are now (the products cannot be put
// off past this point, with the bond's matrix saved for later).
template <int D>
__device__ __forceinline__ void end_bond(double (&H)[D]) {
#pragma unroll
    for (int d = 0; d < D; ++d) asm volatile("" : "+v"(H[d]));
}

// The small LDS tables of a trajectory, `chunk` steps' envelopes and records
// at a time.
struct MixTables {
    double* cst;   // [rows][3]: B, d0, d1 of every field component
    double* hin;   // [2 step parity][4][rows]: the drive at the step's start, -(B + drive) at its middle and end, -B
    double* drv;   // [2 chunk parity][chunk][3 stage times][2 species][2 pulses]
    double* red;   // record sums
    int rows;      // 3 A2 + 8 A3
};

// B, d0, d1 of field component i (the SU(2) sublattices' first).
struct MixRow {
    double B, d0, d1;
};
__device__ __forceinline__ MixRow mix_row(cptr<MixDev> M, int i) {
    const int n2 = 3 * M->A2, n3 = 8 * M->A3;
    const bool f = i < n2;
    const int j = f ? i : i - n2;
    return {f ? M->field2[j] : M->field3[j], f ? M->fdrive2[j] : M->fdrive3[j],
            f ? M->fdrive2[n2 + j] : M->fdrive3[n3 + j]};
}

// cst and the undriven rows
__device__ __forceinline__ void mix_fill_tables(cptr<MixDev> M, const MixTables& Q, int tid, int T) {
    const int R = Q.rows;
    for (int i = tid; i < R; i += T) {
        const MixRow r = mix_row(M, i);
        Q.cst[3 * i] = r.B;
        Q.cst[3 * i + 1] = r.d0;
        Q.cst[3 * i + 2] = r.d1;
        for (int par = 0; par < 2; ++par)  // without a drive the rows stay 0 and -B
            for (int st = 0; st < 4; ++st) Q.hin[(par * 4 + st) * R + i] = st ? -r.B : 0.0;
    }
}

// Envelopes of steps n0 .. n0 + chunk - 1 (at most 5) into chunk buffer cp,
// by one wave: lane = (step, stage time, species, pulse).
__device__ __forceinline__ void mix_write_drive(const MixTables& Q, int b, int n0, int s_end, int cp, int chunk, int lane) {
    if (lane >= 12 * chunk) return;
    const MixArgsP G = mix_kern_args();
    const cptr<MixDev> M = as_const(G->M);
    const int q = lane / 12, st = (lane % 12) >> 2, s3 = (lane >> 1) & 1, kk = lane & 1;
    const int n = n0 + q;
    if (n >= s_end) return;
    const double t = G->A.tgrid[n], dt = G->A.dt;
    const double ts = st == 0 ? t : (st == 1 ? t + 0.5 * dt : t + 1.0 * dt);
    const double amp = s3 ? M->amp3 : M->amp2;
    double v = 0.0;
    if (amp != 0.0) {
        const double tc = (s3 ? G->A.tp3 : G->A.tp)[2 * size_t(b) + kk];
        v = drive_factor(amp, ts, tc, s3 ? M->width3 : M->width2, s3 ? M->freq3 : M->freq2);
        if (G->A.scale) v *= G->A.scale[2 * size_t(b) + kk];
    }
    Q.drv[cp * 12 * chunk + lane] = v;
}

// Field rows 0 to 2 of the step whose envelopes are f[0..11].
__device__ __forceinline__ void mix_write_hin(const MixTables& Q, const double* f, int par, int n2, int tid, int T) {
    const int R = Q.rows;
    for (int i = tid; i < 3 * R; i += T) {
        const int st = i / R, r = i - st * R, s3 = r < n2 ? 0 : 2;
        const double D = Q.cst[3 * r + 1] * f[st * 4 + s3] + Q.cst[3 * r + 2] * f[st * 4 + s3 + 1];
        Q.hin[par * 4 * R + i] = st ? -Q.cst[3 * r] - D : D;
    }
}

// One row st of the one set of rows of the tight layout (csl_mixed_lay.hpp);
// f null: no drive.
__device__ __forceinline__ void mix_write_row(cptr<MixDev> M, const MixTables& Q, const double* f, int st, int n2, int tid,
                                              int T) {
    for (int i = tid; i < Q.rows; i += T) {
        const MixRow r = mix_row(M, i);
        const int s3 = i < n2 ? 0 : 2;
        const double D = f && st < 3 ? r.d0 * f[st * 4 + s3] + r.d1 * f[st * 4 + s3 + 1] : 0.0;
        Q.hin[st * Q.rows + i] = st ? -r.B - D : D;
    }
}

// One record from the units' sums, a lane per value: s2(unit, c) the SU(2)
// sums, s3(unit, c) the SU(3) ones, alt(unit, c) those with the sign of the
// site index when that changes from cell to cell (odd A3), twice_e the sum
// of the energy shares.
template <class F2, class F3, class FA, class FE>
__device__ __forceinline__ void mix_publish(int b, int ri, int lane, F2 s2, F3 s3, FA alt, FE twice_e) {
    const MixArgsP G = mix_kern_args();
    const cptr<MixDev> M = as_const(G->M);
    const int per = M->npad / kWave, A2 = M->A2, A3 = M->A3;
    if (lane >= kRec) return;
    double v = 0.0;
    if (lane < 9) {
        const int g = lane / 3, d = lane % 3;
        for (int at = 0; at < A2; ++at) {
            double s[3] = {0.0, 0.0, 0.0};
            for (int i = 0; i < per; ++i)
                for (int c = 0; c < 3; ++c) s[c] += s2(at * per + i, c);
            const double* Rm = M->frames2 + at * 9 + d * 3;
            const double gl = Rm[0] * s[0] + Rm[1] * s[1] + Rm[2] * s[2];
            const double own = d == 0 ? s[0] : (d == 1 ? s[1] : s[2]);
            v += g == 0 ? M->afm2[at] * gl : (g == 1 ? own : gl);
        }
    } else if (lane < 33) {
        const int g = (lane - 9) / 8, d = (lane - 9) % 8;
        for (int at = 0; at < A3; ++at) {
            double s[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, al = 0.0;
            for (int i = 0; i < per; ++i) {
                for (int c = 0; c < 8; ++c) s[c] += s3(at * per + i, c);
                if (A3 & 1) al += alt(at * per + i, d);
            }
            double own = 0.0, gl = 0.0;
            const double* Rm = M->frames3 + at * 64 + d * 8;
            for (int c = 0; c < 8; ++c) {
                own = c == d ? s[c] : own;
                gl += Rm[c] * s[c];
            }
            v += g == 0 ? ((A3 & 1) ? al : ((at & 1) ? -own : own)) : (g == 1 ? own : gl);
        }
    } else {
        v = 0.5 * twice_e();
    }
    const double sc = lane < 9 ? G->A.inv2 : (lane < 33 ? G->A.inv3 : G->A.invE);
    G->A.recs[(size_t(ri) * G->A.B_rec + b) * kRec + lane] = v * sc;
}

// The rows of a work-split schedule (or trajectory piece * grid + block):
// false when this workgroup has no further piece.
struct MixPiece {
    int b, s_begin, s_end, wait, post;
};
__device__ __forceinline__ bool mix_piece(const MixPersistArgs& A, int piece, MixPiece& P) {
    P = {int(blockIdx.x) + piece * int(gridDim.x), 0, A.n_steps, -1, -1};
    if (A.sched) {
        if (piece >= A.max_pieces) return false;
        const int* r = A.sched + (size_t(blockIdx.x) * A.max_pieces + piece) * 5;
        P = {uniform(r[0]), uniform(r[1]), uniform(r[2]), uniform(r[3]), uniform(r[4])};
        if (P.b < 0) return false;  // unused rows come last
    } else if (P.b >= A.B) {
        return false;
    }
    P.b += A.b0;
    return true;
}

// Waits for the state of a seam, stored in X by the workgroup that ran the
// trajectory's first steps as its first piece; a bounded wait that gives up
// flags the launch.  Called by every thread.
__device__ __forceinline__ void mix_wait_seam(const MixPersistArgs& A, int wait, int tid) {
    if (tid == 0) {
        unsigned ok = 0;
        for (long it = 0; it < (1L << 24); ++it) {
            ok = __hip_atomic_load(A.flags + wait, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
            if (ok) break;
            __builtin_amdgcn_s_sleep(8);
        }
        if (!ok) __hip_atomic_store(A.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
}

}  // namespace

}  // namespace csl
