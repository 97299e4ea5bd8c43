"""Every variant of the mixed lattice's persistent kernels, told by last_path():
SU(3)-SU(3) bonds, onsite matrices, fields, frames, Gilbert and Bloch damping
and pulses at each size class (one unit of 64 sites per wave; two to four units
a wave with SU(3) components 6 and 7 in LDS or in device memory), odd numbers
of SU(3) sublattices (whose staggered sign changes from cell to cell), and the
tangent run beyond the packed tables' 2048 sites and with per-site matrices.

Tolerances as in test_gpu_mixed_shapes.py: some 100 roundings a step and
component, 1e-12 for the few steps here (the onsite matrices and damping add
less than half as many again).  Tangents against central differences as in
test_gpu_mixed_grad.py.
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import gpu_mixed as GM
from classical_mcmc_spin_amd import mixed_model as mm
from test_gpu_mixed_uneven import uneven_cell
from test_mixed_oracle import random_flat, rich_cell

pytestmark = pytest.mark.gpu

DT = 0.005


def _against_oracle(oracle, muc, dims, steps, every, want, seed=5):
    ml = mm.MixedLattice(muc, *dims)
    A2, A3 = ml.su2.N_atoms, ml.su3.N_atoms
    g = np.random.default_rng(seed)
    init = random_flat(ml, seed)
    f2, f3 = g.normal(size=(A2, 3)), g.normal(size=(A3, 8))
    gamma = np.array([0.05, 0.0, 0.02, 0.0, 0.03, 0.0, 0.0, 0.01])
    eq = 0.1 * g.normal(size=(ml.N3, 8))
    tp = np.array([[0.0, 0.01], [0.01, 0.0]])
    sc = np.array([[1.0, 0.5], [0.0, 1.0]])
    T1 = (steps + 0.5) * DT
    print(f"[mixed variant] {A2} + {A3} x {dims} {want}", flush=True)
    with GM.GPUMixedLattice(ml) as gm:
        gm.set_damping(0.03, gamma, eq)
        GM._set_pulses(gm, f2, f2, f3, f3, 0.0, 0.0, 0.5, 0.02, 3.0, 0.4, 0.03, 0.0)
        r = gm.integrate_batched(init, tp, sc, 0.0, T1, DT, save_interval=every, want_final=True)
        path = gm.last_path()
    assert path["persistent"]
    assert tuple(path[k] for k in ("unit_waves", "global_67", "tight")) == want
    keep = sorted(set(range(0, steps, every)) | {steps})
    for b in range(2):
        o = oracle.MixedOracle(muc, *dims)
        o.set_damping(0.03, gamma, eq)
        o.set_pulse(2, f2 * sc[b, 0], tp[b, 0], f2 * sc[b, 1], tp[b, 1], 0.5, 0.02, 3.0)
        o.set_pulse(3, f3 * sc[b, 0], tp[b, 0], f3 * sc[b, 1], tp[b, 1], 0.4, 0.03, 0.0)
        ref = o.integrate_md(init, 0.0, T1, DT)
        assert np.max(np.abs(r["records"][:, b] - ref["records"][keep])) <= 1e-12
        assert np.max(np.abs(r["final"][b] - ref["final"])) <= 1e-12


WAVES, LDS, GLOBAL, TIGHT = (True, False, False), (False, False, False), (False, True, False), (False, True, True)


@pytest.mark.parametrize("dims,steps,every,want", [
    ((3, 2, 2), 6, 1, WAVES), ((5, 5, 3), 3, 2, WAVES),
    ((6, 5, 5), 5, 1, LDS),      # two units a wave
    ((7, 7, 6), 3, 1, LDS),      # three
    ((8, 8, 7), 3, 1, GLOBAL),   # four
    ((8, 8, 8), 4, 3, GLOBAL),
])
def test_su3_bonds(oracle, dims, steps, every, want):
    _against_oracle(oracle, rich_cell(), dims, steps, every, want)


@pytest.mark.parametrize("A2,A3,dims,tt,want", [
    (4, 3, (3, 3, 3), False, WAVES), (4, 3, (8, 8, 5), False, LDS), (3, 3, (10, 8, 8), False, GLOBAL),
    (2, 1, (5, 5, 5), True, WAVES), (4, 3, (8, 8, 5), True, LDS), (3, 3, (10, 8, 8), True, GLOBAL),
    (24, 24, (4, 4, 4), True, GLOBAL),     # three units a wave, components 6 and 7 in device memory
    (16, 15, (5, 5, 5), True, TIGHT), (32, 32, (4, 4, 4), False, TIGHT),
])
def test_sublattice_counts(oracle, A2, A3, dims, tt, want):
    _against_oracle(oracle, uneven_cell(A2, A3, tt), dims, 3, 1, want)


@pytest.mark.parametrize("damped", [False, True])
def test_tangent_beyond_the_packed_tables(oracle, damped):
    """2304 sites of each species: the counted loops over the bond tables."""
    muc, dims, n, h = rich_cell(), (9, 8, 8), 4, 1e-5
    ml = mm.MixedLattice(muc, *dims)
    init = random_flat(ml, 3)
    gamma, eq = np.full(8, 0.02), np.zeros((ml.N3, 8))
    T1 = (n + 0.5) * DT

    def run(scale):
        o = oracle.MixedOracle(mm.scale_fe_tm(muc, scale), *dims)
        if damped:
            o.set_damping(0.03, gamma, eq)
        return o.integrate_md(init, 0.0, T1, DT)["records"]

    ref, fd = run(1.0), (run(1.0 + h) - run(1.0 - h)) / (2.0 * h)
    with GM.GPUMixedLattice(ml) as gm:
        if damped:
            gm.set_damping(0.03, gamma, eq)
        g = gm.scale_gradient(init, [[0.0, 0.0]], ref + 0.01, np.r_[np.ones(33), 0.0], None, 0.0, T1, DT,
                              want_records=True)
    assert np.max(np.abs(g["records"][:, 0] - ref)) <= 1e-12
    assert np.max(np.abs(g["trecords"][:, 0, :33] - fd[:, :33])) <= 1e-6 * np.max(np.abs(fd[:, :33]))


def test_tangent_with_matrices_of_every_site():
    """Mixed and SU(2) matrices that differ from site to site, against central
    differences of the device's forward run (stage kernels)."""
    dims, n, h = (3, 2, 2), 8, 1e-5
    g = np.random.default_rng(2)

    def lattice(scale):
        ml = mm.MixedLattice(rich_cell(), *dims)
        g = np.random.default_rng(2)
        f = 1.0 + 0.3 * g.normal(size=(ml.N2, ml.N3))          # the factor of a mixed bond, the same from both sides
        i2 = np.repeat(np.arange(ml.N2), np.diff(ml.m2_offset.astype(int)))
        i3 = np.repeat(np.arange(ml.N3), np.diff(ml.m3_offset.astype(int)))
        ml.m2_J = ml.m2_J * (scale * f[i2, ml.m2_partner.astype(int)])[:, None, None]
        ml.m3_J = ml.m3_J * (scale * f[ml.m3_partner.astype(int), i3])[:, None, None]
        return ml

    T1 = (n + 0.5) * DT
    init = random_flat(lattice(1.0), 4)

    def run(scale):
        with GM.GPUMixedLattice(lattice(scale)) as gm:
            r = gm.integrate_batched(init, [[0.0, 0.0]], None, 0.0, T1, DT)["records"][:, 0]
            assert not gm.last_path()["persistent"]
            return r

    ref, fd = run(1.0), (run(1.0 + h) - run(1.0 - h)) / (2.0 * h)
    with GM.GPUMixedLattice(lattice(1.0)) as gm:
        t = gm.scale_gradient(init, [[0.0, 0.0]], ref, np.r_[np.ones(33), 0.0], None, 0.0, T1, DT, want_records=True)
    assert np.array_equal(t["records"][:, 0], ref)
    assert np.max(np.abs(t["trecords"][:, 0, :33] - fd[:, :33])) <= 1e-6 * np.max(np.abs(fd[:, :33]))
