"""Mixed persistent kernels at the edges of their shapes against the mixed
oracle: the one-unit-per-wave kernel (up to 16 units of 64 sites, nearly
empty and full last units), the kernel of larger lattices with SU(3)
components 6 and 7 in LDS and in global memory, step counts around the chunk
of steps whose records go together, record intervals, one and both pulses.

Tolerance: a step rounds a component some hundred times (eight 8-component
bonds, the structure-constant products, the updates), so 9 steps of unit
vectors differ by at most 9 * 100 * 2.2e-16 = 2e-13 from another order of the
same sums; 1e-12 allows for the growth over the run.
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import gpu_mixed as GM
from classical_mcmc_spin_amd import mixed_model as mm
from classical_mcmc_spin_amd import seeding

pytestmark = pytest.mark.gpu

TOL = 1e-12
DT = 0.005


@pytest.mark.parametrize("dims,steps,every", [
    ((2, 2, 2), 1, 1), ((3, 1, 2), 9, 1), ((4, 4, 4), 4, 1), ((5, 5, 5), 9, 2), ((5, 3, 5), 7, 5),   # one unit per wave
    ((6, 6, 5), 5, 1), ((6, 7, 6), 9, 2),        # larger lattices, all components in LDS
    ((7, 8, 8), 3, 1),                           # components 6, 7 in global memory
])
def test_mixed_shapes(oracle, dims, steps, every):
    muc = mm.build_tmfeo3_mixed()
    ml = mm.MixedLattice(muc, *dims)
    g = ml.flat_state(seeding.random_spins(ml.N2, 5), mm.random_su3_states(ml.N3, 6))
    f2, f3 = np.zeros((4, 3)), np.zeros((4, 8))
    f2[:, 0], f3[:, 1] = 1.0, 1.0
    tp = np.array([[0.0, 0.0], [0.01, 0.02], [0.0, 0.03]])
    sc = np.array([[0.0, 0.0], [1.0, 0.5], [0.0, 1.0]])
    T1 = (steps + 0.5) * DT
    print(f"[mixed] {dims} steps {steps} every {every}", flush=True)
    gm = GM.GPUMixedLattice(ml)
    try:
        GM._set_pulses(gm, f2, f2, f3, f3, 0.0, 0.0, 0.5, 0.02, 3.0, 0.4, 0.03, 0.0)
        r = gm.integrate_batched(g, tp, sc, 0.0, T1, DT, save_interval=every, want_final=True)
        assert gm.last_path()["persistent"]
    finally:
        gm.close()
    keep = sorted(set(range(0, steps, every)) | {steps})
    assert r["records"].shape[0] == len(keep)
    for b in range(3):
        o = oracle.MixedOracle(muc, *dims)
        o.set_pulse(2, f2 * sc[b, 0], tp[b, 0], f2 * sc[b, 1], tp[b, 1], 0.5, 0.02, 3.0)
        o.set_pulse(3, f3 * sc[b, 0], tp[b, 0], f3 * sc[b, 1], tp[b, 1], 0.4, 0.03, 0.0)
        ref = o.integrate_md(g, 0.0, T1, DT)
        assert np.max(np.abs(r["records"][:, b] - ref["records"][keep])) <= TOL
        assert np.max(np.abs(r["final"][b] - ref["final"])) <= TOL
