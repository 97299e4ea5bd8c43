"""Mixed lattices whose species have different numbers of sublattices: the
packed partner tables of the tangent run (their unused slots on the host:
test_mixed_pack.py).

Tolerances: runs against the oracle as in test_gpu_mixed_shapes.py (some 100
roundings a step and component, 1e-12 for up to 9 steps of unit vectors); the
tangent records against central differences of the oracle's runs at scales
1 +- 1e-5 (truncation 1e-10, rounding 1e-16 / 1e-5 a record) to 1e-6 of their
largest, as in test_gpu_mixed_grad.py.
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import gpu_mixed as GM
from classical_mcmc_spin_amd import mixed_model as mm
from classical_mcmc_spin_amd import seeding
from classical_mcmc_spin_amd.model import UnitCell

pytestmark = pytest.mark.gpu

DT = 0.005


def uneven_cell(A2, A3, tt=False, seed=7):
    """A2 SU(2) and A3 SU(3) sublattices, fields and onsite terms of both;
    four SU(2) bonds a sublattice, two mixed bonds a SU(2) sublattice, and with
    tt SU(3)-SU(3) bonds of the first sublattice."""
    g = np.random.default_rng(seed)
    fe, tm = UnitCell(3, A2), UnitCell(8, A3)
    sym = lambda n, s: (lambda m: s * (m + m.T))(g.normal(size=(n, n)))
    for a in range(A2):
        fe.set_field(0.2 * g.normal(size=3), a)
        fe.set_onsite_interaction(sym(3, 0.05), a)
        for o in ((0, 0, 0), (0, 0, 1)):
            fe.set_bilinear_interaction(0.3 * g.normal(size=(3, 3)), a, (a + 1) % A2, o)
    fe.set_afm_sublattice_signs(np.where(np.arange(A2) % 2, -1.0, 1.0))
    for a in range(A3):
        tm.set_field(0.3 * g.normal(size=8), a)
        tm.set_onsite_interaction(sym(8, 0.05), a)
    if tt:
        tm.set_bilinear_interaction(0.1 * g.normal(size=(8, 8)), 0, A3 - 1, (0, 0, 1))
    muc = mm.MixedUnitCell(fe, tm)
    for a in range(A2):
        for o in ((0, 0, 0), (0, 1, 0)):
            muc.set_mixed_bilinear(0.2 * g.normal(size=(3, 8)), a, a % A3, o)
    return muc


@pytest.mark.parametrize("A2,A3,dims,tt", [(4, 2, (3, 2, 2), False), (2, 3, (5, 3, 5), True), (6, 1, (1, 5, 2), False)])
def test_tangent_with_uneven_sublattices(oracle, A2, A3, dims, tt):
    muc = uneven_cell(A2, A3, tt)
    ml = mm.MixedLattice(muc, *dims)
    init = ml.flat_state(seeding.random_spins(ml.N2, 3), mm.random_su3_states(ml.N3, 4))
    n = 12
    T1 = (n + 0.5) * DT
    w = np.r_[np.ones(33), 0.0]
    run = lambda s: oracle.MixedOracle(mm.scale_fe_tm(muc, s), *dims).integrate_md(init, 0.0, T1, DT)["records"]
    ref = run(1.0)
    h = 1e-5
    fd = (run(1.0 + h) - run(1.0 - h)) / (2.0 * h)
    target = ref + 0.01
    with GM.GPUMixedLattice(ml) as gm:
        g = gm.scale_gradient(init, [[0.0, 0.0]], target, w, None, 0.0, T1, DT, want_records=True)
    assert np.max(np.abs(g["records"][:, 0] - ref)) <= 1e-12
    tr = g["trecords"][:, 0]
    assert np.max(np.abs(tr[:, :33] - fd[:, :33])) <= 1e-6 * np.max(np.abs(fd[:, :33]))
    grad = 2.0 * np.sum(w * (ref - target) * tr)
    # 33 n products of records within 1e-12 and these tangents, summed in another order
    assert abs(g["grad"][0] - grad) <= 1e-10 * np.sum(np.abs(w * (ref - target) * tr))


@pytest.mark.parametrize("A2,A3,dims,tt,steps,every", [
    (16, 16, (8, 4, 4), True, 5, 1),      # 128 cells: 170 KB with the roomy tables
    (16, 16, (5, 5, 5), False, 4, 3),
    (32, 31, (4, 4, 4), False, 3, 1),     # 64 cells, the most sublattices; odd
    (32, 31, (1, 9, 7), True, 2, 2),
])
def test_many_sublattices_stay_persistent(oracle, A2, A3, dims, tt, steps, every):
    """Lattices of 2048 sites of each species whose field rows leave no room
    for two steps' worth: driven, three trajectories, against the oracle."""
    muc = uneven_cell(A2, A3, tt)
    ml = mm.MixedLattice(muc, *dims)
    init = ml.flat_state(seeding.random_spins(ml.N2, 3), mm.random_su3_states(ml.N3, 4))
    g = np.random.default_rng(1)
    f2, f3 = g.normal(size=(A2, 3)), g.normal(size=(A3, 8))
    tp = np.array([[0.0, 0.0], [0.01, 0.015], [0.0, 0.02]])
    sc = np.array([[0.0, 0.0], [1.0, 0.5], [0.0, 1.0]])
    T1 = (steps + 0.5) * DT
    print(f"[mixed] {A2} + {A3} sublattices of {dims}", flush=True)
    with GM.GPUMixedLattice(ml) as gm:
        GM._set_pulses(gm, f2, f2, f3, f3, 0.0, 0.0, 0.5, 0.02, 3.0, 0.4, 0.03, 0.0)
        r = gm.integrate_batched(init, tp, sc, 0.0, T1, DT, save_interval=every, want_final=True)
        assert gm.last_path()["persistent"]
    keep = sorted(set(range(0, steps, every)) | {steps})
    for b in range(3):
        o = oracle.MixedOracle(muc, *dims)
        o.set_pulse(2, f2 * sc[b, 0], tp[b, 0], f2 * sc[b, 1], tp[b, 1], 0.5, 0.02, 3.0)
        o.set_pulse(3, f3 * sc[b, 0], tp[b, 0], f3 * sc[b, 1], tp[b, 1], 0.4, 0.03, 0.0)
        ref = o.integrate_md(init, 0.0, T1, DT)
        assert np.max(np.abs(r["records"][:, b] - ref["records"][keep])) <= 1e-12
        assert np.max(np.abs(r["final"][b] - ref["final"])) <= 1e-12


@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 3, 3), (7, 7, 5), (8, 8, 8)])
@pytest.mark.parametrize("coupled", [False, True])
def test_an_overflow_stays_where_the_bonds_lead(dims, coupled):
    """SU(3) sites that overflow (values of 1e200 at the start) leave alone what
    no bond ties to them: the SU(2) species without mixed bonds, or with them
    the SU(3) sublattice that has none.  The same states to the last bit as
    beside ordinary spins, in the batch and in the tangent run's forward one."""
    muc = uneven_cell(4, 3)
    # mixed bonds to the first two SU(3) sublattices, or none
    muc.bilinear_SU2_SU3 = [b for b in muc.bilinear_SU2_SU3 if b.partner < 2] if coupled else []
    ml = mm.MixedLattice(muc, *dims)
    s2, s3 = seeding.random_spins(ml.N2, 3), mm.random_su3_states(ml.N3, 4)
    huge = s3.copy()
    wild = np.arange(ml.N3) % 3 != 2 if coupled else np.ones(ml.N3, bool)
    huge[wild] *= 1e200
    n = 3
    T1 = (n + 0.5) * DT
    out = []
    with GM.GPUMixedLattice(ml) as gm:
        for x in (s3, huge):
            init = ml.flat_state(s2, x)
            r = gm.integrate_batched(init, [[0.0, 0.0]], None, 0.0, T1, DT, want_final=True)
            assert gm.last_path()["persistent"]
            g = gm.scale_gradient(init, [[0.0, 0.0]], np.zeros((n + 1, 34)), np.r_[np.ones(33), 0.0], None, 0.0, T1,
                                  DT, want_records=True)
            out.append((ml.split_state(r["final"][0]), r["records"][:, 0], g["records"][:, 0], g["trecords"][:, 0]))
    (a2, a3), (b2, b3) = out[0][0], out[1][0]
    assert not np.all(np.isfinite(b3))
    if coupled:
        assert np.array_equal(a3[~wild], b3[~wild])
    else:
        assert np.array_equal(a2, b2)
        for q in (1, 2):
            assert np.array_equal(out[0][q][:, :9], out[1][q][:, :9])
        assert np.all(out[1][3][:, :9] == 0.0)
