"""The atom-major persistent kernel (k_trajectory) at the edges of its tiles
and chunks against the oracle: lattices whose last unit of 64 cells is nearly
empty or exactly full, 3, 6 and 12 bonds per site, 2 and 16 sublattices,
damping, step counts around the chunk of 8 steps and record intervals below,
at and above it.

Tolerance: a step rounds each component some thirty times (27 bond products,
the cross product, the updates), so 41 steps of unit spins stay within
41 * 30 * 2.2e-16 = 3e-13 of another order of the same sums; 1e-12 allows for
the growth along the trajectory (less than a factor of two over 0.41 units of
time).
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import GPULattice, model
from helpers import random_state

pytestmark = pytest.mark.gpu

TOL = 1e-12
DT = 0.01


def _kitaev(**kw):
    return model.build_kitaev_honeycomb(field_strength=0.1, field_direction=(1.0, 1.0, 1.0), **kw)


CELLS = {
    "z3_5x3": (lambda: _kitaev(), (5, 3, 1)),            # 15 of 64 cells
    "z3_8x8": (lambda: _kitaev(), (8, 8, 1)),            # one full unit
    "z3_13x5": (lambda: _kitaev(), (13, 5, 1)),          # 65 cells: a second unit with one cell
    "z3_23x25": (lambda: _kitaev(), (23, 25, 1)),        # 9 units over uneven waves
    "z12_6x7": (lambda: _kitaev(J2_A=0.1, J2_B=-0.07, J3=0.05), (6, 7, 1)),
    "z6_pyro2": (lambda: model.build_pyrochlore_conventional(field_strength=0.1), (2, 2, 2)),
}


@pytest.mark.parametrize("name", sorted(CELLS))
@pytest.mark.parametrize("steps,every,alpha", [(1, 1, 0.0), (8, 1, 0.03), (41, 1, 0.0), (41, 3, 0.0), (23, 11, 0.03)])
def test_trajectory_edges(oracle, name, steps, every, alpha):
    build, dims = CELLS[name]
    uc = build()
    lat = model.Lattice(uc, *dims)
    s = random_state(lat, 77)
    f = np.zeros((lat.N_atoms, 3))
    f[:, 0] = 1.0
    fd = np.einsum("aij,aj->ai", lat.frames, f).reshape(-1)
    T1 = (steps + 0.5) * DT
    tp = np.array([[0.0, 0.2], [0.1, 0.0], [0.0, 0.0]])
    am = np.array([[0.5, 0.25], [0.5, 0.0], [0.0, 0.0]])
    print(f"[trajectory] {name} steps {steps} every {every} alpha {alpha}", flush=True)
    with GPULattice(lat) as gl:
        gl.set_damping(alpha)
        gl.set_pulse(np.concatenate([fd, fd]), 0.5, 0.1, 3.0, 0.0, 0.0)
        r = gl.integrate_batched(s, tp, am, 0.0, T1, DT, save_interval=every, tgrid="boost", want_final=True)
        assert gl.last_launch_config()["atom_major"]
    o = oracle.OracleLattice(uc, *dims)
    o.set_alpha(alpha)
    keep = sorted(set(range(0, steps, every)) | {steps})
    for b in range(3):
        o.set_pulse(f * (am[b, 0] / 0.5), tp[b, 0], f * (am[b, 1] / 0.5), tp[b, 1], 0.5, 0.1, 3.0)
        ref = o.integrate_md(s.reshape(-1), 0.0, T1, DT)
        assert r["mags"].shape[0] == len(keep)
        assert np.max(np.abs(r["mags"][:, b] - ref["mags"][keep])) <= TOL
        assert np.max(np.abs(r["energy"][:, b] - ref["energy"][keep])) <= TOL
        assert np.max(np.abs(r["final"][b] - ref["final"].reshape(-1, 3))) <= TOL


@pytest.mark.parametrize("dims,shapes", [((23, 25, 1), {2, 3}), ((36, 28, 1), {2, 3, 4, 6}), ((31, 39, 1), {3, 4})])
@pytest.mark.parametrize("alpha", [0.0, 0.03])
def test_twelve_bonds_every_sites_per_thread(oracle, dims, shapes, alpha):
    """Twelve bonds a site, damped and not, at every atom-major launch shape of
    the lattice (from three sites a thread on the partners are packed)."""
    uc = _kitaev(J2_A=0.1, J2_B=-0.07, J3=0.05)
    lat = model.Lattice(uc, *dims)
    s = random_state(lat, 78)
    steps = 9
    T1 = (steps + 0.5) * DT
    o = oracle.OracleLattice(uc, *dims)
    o.set_alpha(alpha)
    ref = o.integrate_md(s.reshape(-1), 0.0, T1, DT)
    seen = set()
    with GPULattice(lat) as gl:
        gl.set_damping(alpha)
        for c in gl.launch_candidates():
            if not c["atom_major"]:
                continue
            gl.set_launch_config(2, c["block"], c["sites_per_thread"], c["flags"])
            print(f"[twelve] {dims} alpha {alpha} {c}", flush=True)
            r = gl.integrate_batched(s, np.zeros((2, 2)), np.zeros((2, 2)), 0.0, T1, DT, tgrid="boost", want_final=True)
            assert gl.last_launch_config()["atom_major"]
            seen.add(c["sites_per_thread"])
            for b in range(2):
                assert np.max(np.abs(r["mags"][:, b] - ref["mags"])) <= TOL
                assert np.max(np.abs(r["energy"][:, b] - ref["energy"])) <= TOL
                assert np.max(np.abs(r["final"][b] - ref["final"].reshape(-1, 3))) <= TOL
    assert shapes <= seen


@pytest.mark.parametrize("n_tau,steps", [(1, 1), (7, 15), (8, 16), (17, 33)])
def test_pump_probe_rows(n_tau, steps):
    """Trajectory-major pump-probe records (tiles of 16 records x 16
    trajectories) are the batch's own records, the start sample dropped."""
    lat = model.Lattice(_kitaev(), 5, 4, 1)
    s = random_state(lat, 3)
    f = np.zeros((2, 3))
    f[:, 0] = 1.0
    T1 = -0.1 + (steps + 0.5) * DT
    print(f"[pump] n_tau {n_tau} steps {steps}", flush=True)
    with GPULattice(lat) as gl:
        r = gl.pump_probe(s, f, 0.5, 0.1, 0.0, 0.0, 0.02 * (n_tau - 0.5), 0.02, -0.1, T1, DT)
        fd = np.einsum("aij,aj->ai", lat.frames, f).reshape(-1)
        gl.set_pulse(np.concatenate([fd, fd]), 0.5, 0.1, 0.0, 0.0, 0.0)
        taus = 0.02 * np.arange(n_tau)
        B = 1 + 2 * n_tau
        tp, am = np.zeros((B, 2)), np.zeros((B, 2))
        am[0, 0] = 0.5
        tp[1:1 + n_tau, 0], am[1:1 + n_tau, 0] = taus, 0.5
        tp[1 + n_tau:, 1], am[1 + n_tau:] = taus, 0.5
        b = gl.integrate_batched(s, tp, am, -0.1, T1, DT, tgrid="boost")
    m = b["mags"][1:]
    assert r["M0"].shape == (steps, 3, 3) and r["M1"].shape == r["M01"].shape == (n_tau, steps, 3, 3)
    assert np.array_equal(r["times"], b["times"][1:])
    assert np.array_equal(r["M0"], m[:, 0])
    assert np.array_equal(r["M1"], np.swapaxes(m[:, 1:1 + n_tau], 0, 1))
    assert np.array_equal(r["M01"], np.swapaxes(m[:, 1 + n_tau:], 0, 1))


@pytest.mark.parametrize("step,steps,kept", [(1e-10, 4, 5), (1.0000001e-10, 4, 4), (2.5e-11, 7, 8)])
def test_pump_probe_keeps_the_start_of_fine_grids(step, steps, kept):
    """The observer gate passes a sample less than 1e-10 short of a step after
    the last one: the start sample too where the step is that fine."""
    lat = model.Lattice(_kitaev(), 3, 2, 1)
    f = np.zeros((2, 3))
    f[:, 0] = 1.0
    with GPULattice(lat) as gl:
        r = gl.pump_probe(random_state(lat, 3), f, 0.5, 0.1, 0.0, 0.0, 0.02, 0.02, 0.0, (steps + 0.5) * step, step)
    assert r["M0"].shape == (kept, 3, 3) and r["M1"].shape[:2] == r["M01"].shape[:2] == (2, kept)
    t = step * np.arange(steps + 1)
    assert np.array_equal(r["times"], t[steps + 1 - kept:])


@pytest.mark.parametrize("dims,steps,every", [((5, 3, 1), 19, 1), ((13, 5, 1), 24, 8), ((4, 6, 1), 37, 5)])
@pytest.mark.parametrize("onsite", [0.0, 0.1])
def test_structure_factor_samples(dims, steps, every, onsite):
    """Samples left by the persistent kernels (atom-major, and the general
    one for an onsite matrix) and their batched transforms against numpy on
    the stage engine's states.  The power sums |S(q, w)|^2 of some thousand
    rounded terms: 1e-12 relative to the largest."""
    lat = model.Lattice(_kitaev(Ka=onsite, Kb=-onsite, Kc=0.5 * onsite), *dims)
    B, n_t = 3, steps // every
    T1 = (steps + 0.5) * DT
    init = np.stack([random_state(lat, 40 + b) for b in range(B)])
    pos = np.array([[0.0, 0.0, 0.0], [0.1, 0.55, 0.0]])
    print(f"[dssf] {dims} steps {steps} every {every} onsite {onsite}", flush=True)
    states = []
    with GPULattice(lat) as gl:
        r = gl.structure_factor(init, 0.0, T1, DT, every, dims, pos, want_mags=True)
        for b in range(B):
            gl.set_spins(init[b])
            states.append(gl.integrate(0.0, T1, DT, tgrid="boost", engine=1, want_states=True)["states"])
    S = np.stack(states, 1)[:-1:every][:n_t]                       # [n_t, B, N, 3]
    F = np.fft.fftn(S.reshape((n_t, B) + dims + (2, 3)), axes=(2, 3, 4))
    q = np.stack(np.meshgrid(*[2 * np.pi * np.arange(L) / L for L in dims], indexing="ij"), -1)
    ph = np.exp(-1j * np.einsum("ijkc,ac->ijka", q, pos))
    sw = np.fft.fft((F * ph[..., None]).sum(-2), axis=0)
    p = (np.abs(sw) ** 2).sum((1, 5)) / (B * lat.lattice_size * n_t)
    ref = p.reshape(n_t, -1).T
    assert r["sqw"].shape == ref.shape
    assert np.max(np.abs(r["sqw"] - ref)) <= 1e-12 * np.max(ref)
    m = S.mean(2)
    assert np.max(np.abs(r["mags"][:-1:every][:n_t, :, 1] - m)) <= 1e-13


@pytest.mark.parametrize("B,n_t,kept", [(4, 30, True), (128, 1200, False)])
def test_structure_factor_buffers(B, n_t, kept):
    """A call repeated on its handle gives the same bits, also with a call of
    another shape between; buffers of up to 8 GB stay on the handle, larger
    ones (samples and S(q, t) 4.2 GB each here) are given back."""
    import torch
    lat = model.Lattice(_kitaev(), 24, 24, 1)
    init = np.stack([random_state(lat, b) for b in range(B)])
    pos = np.array([[0.0, 0.0, 0.0], [0.1, 0.55, 0.0]])

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    with GPULattice(lat) as gl:
        run = lambda n: gl.structure_factor(init, 0.0, (n + 0.5) * DT, DT, 1, (24, 24, 1), pos)["sqw"]
        gl.integrate_batched(init, np.zeros((B, 2)), np.zeros((B, 2)), 0.0, (n_t + 0.5) * DT, DT, tgrid="boost")
        before = used()
        first = run(n_t)
        held = used() - before
        print(f"[dssf buffers] B {B} samples {n_t}: {held / 2**20:.0f} MB stay", flush=True)
        samples = 8 * n_t * B * lat.lattice_size * 3
        assert (held >= samples) if kept else (held < 64 << 20)
        second = run(n_t)
        run(n_t // 2)
        third = run(n_t)
    assert np.array_equal(first, second) and np.array_equal(first, third)
