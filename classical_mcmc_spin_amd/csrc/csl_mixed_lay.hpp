// csl_mixed_lay.hpp — LDS layout of the mixed lattice's persistent kernel
// (csl_mixed_persist.hip), used by the kernel and its launcher (no HIP).
#pragma once

namespace csl {

constexpr int kMixLdsDoubles = 160 * 1024 / 8;

// Offsets in doubles.  GLDS: SU(3) components 6 and 7 in LDS too.
struct MixPersistLay {
    int chunk = 2;                           // steps whose records and envelopes go together
    bool tight = false;
    // SU(3) [NP3 + 1][6] (and [NP3 + 1][2] with GLDS), SU(2) [NP2 + 1][3]; the
    // last record of each is zero (csl_mixed_pack.hpp)
    int t = 0, t2 = 0, f = 0;
    int cst = 0, hin = 0, drv = 0, red = 0;  // per-sublattice B, d0, d1; field rows; envelopes; record sums
    int rows = 0, n2 = 0, n3 = 0, rec = 0;   // field components; units of each species; doubles per record
    int total = 0;
    // tight: the tables of lattices with many sublattices, 4 doubles a field
    // component instead of 11: B, d0 and d1 stay in device memory, the rows of
    // one step are kept instead of two steps', and records and envelopes go
    // step by step.  Beside 2048 sites of each species 88 bytes a component
    // leave room for 100 components (nine sublattices of each species).  16 + 16
    // sublattices of 128 cells, 256 trajectories x 64 steps: 8.9 ms a call, 11.6
    // on the stage kernels.
    constexpr MixPersistLay(int NP2, int NP3, int A2, int A3, int nwaves, bool glds, bool tight_) : tight(tight_) {
        chunk = tight ? 1 : 2;
        t2 = 6 * (NP3 + 1);
        f = t2 + (glds ? 2 * (NP3 + 1) : 0);
        rows = 3 * A2 + 8 * A3;
        cst = f + 3 * (NP2 + 1);
        cst += cst & 1;
        hin = cst + (tight ? 0 : 3 * rows);
        drv = hin + (tight ? 4 : 8) * rows;
        red = drv + 2 * chunk * 12;
        n2 = NP2 / 64;
        n3 = NP3 / 64;
        // a record: SU(2) units x 4, SU(3) units x 8 (twice with signed
        // sums), one energy sum per wave
        rec = 4 * n2 + ((A3 & 1) ? 16 : 8) * n3 + 4 * nwaves;
        total = red + chunk * rec;
    }
};

// The layout a lattice takes: tight where the other does not fit.
constexpr MixPersistLay mix_persist_lay(int NP2, int NP3, int A2, int A3, int nwaves, bool glds) {
    const MixPersistLay Y(NP2, NP3, A2, A3, nwaves, glds, false);
    return Y.total <= kMixLdsDoubles ? Y : MixPersistLay(NP2, NP3, A2, A3, nwaves, glds, true);
}

}  // namespace csl
