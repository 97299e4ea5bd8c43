"""The adjoint's general backward sweep (k_adj_bwd, k_adj_par and their second
stream), which lattices take that the sweep with register sums does not: six
bonds a site, onsite matrices, a field of every site.

Bar: gradients of a common scale of the bonds and of a uniform field against
central differences of the device's own loss (step 1e-6 of order-one
parameters: truncation 1e-12, rounding of the loss 1e-16 / 1e-6 of it) to 1e-6
of the largest; the loss against the oracle's records to 1e-10 where the
oracle builds the lattice; checkpoint spacings bit for bit.
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import adjoint as AD
from classical_mcmc_spin_amd import model
from classical_mcmc_spin_amd.gpu import GPULattice
from helpers import random_state

pytestmark = pytest.mark.gpu

DT = 0.01
W = np.array([0.5, 0.2, 0.1, 0, 0, 0.3, 1.0, 1.0, 1.0])


def _uc(kind):
    if kind == "pyrochlore":
        return model.build_pyrochlore_conventional(field_strength=0.1)
    J3 = 0.07 if kind == "six" else 0.0
    uc = model.build_kitaev_honeycomb(field_strength=0.1, field_direction=(1.0, 1.0, 1.0), J3=J3)
    if kind == "onsite":
        for a in range(2):
            uc.set_onsite_interaction(np.diag([0.1, -0.05, 0.02 * (a + 1)]), a)
    return uc


def _lattice(kind, dims, jscale=1.0, dh=0.0):
    lat = model.Lattice(_uc(kind), *dims)
    if kind == "site field":
        lat.field = lat.field + 0.1 * np.random.default_rng(6).normal(size=lat.field.shape)
    lat.bi_J = np.ascontiguousarray(lat.bi_J * jscale)
    lat.field = np.ascontiguousarray(lat.field + dh * np.array([0.3, -0.2, 1.0]))
    return lat


@pytest.mark.parametrize("kind,dims", [("pyrochlore", (2, 2, 2)), ("six", (5, 4, 1)), ("six", (13, 9, 1)),
                                       ("onsite", (6, 6, 1)), ("onsite", (16, 20, 1)), ("site field", (9, 8, 1))])
@pytest.mark.parametrize("alpha", [0.0, 0.03])
def test_general_sweep(oracle, kind, dims, alpha):
    n = 33
    T1 = (n + 0.5) * DT
    lat0 = _lattice(kind, dims)
    N, A = lat0.lattice_size, lat0.N_atoms
    init = random_state(lat0, 12)
    target = 0.1 * np.random.default_rng(3).normal(size=(n + 1, 9))
    f = np.zeros((A, 3))
    f[:, 0] = 1.0
    amp, tc = 0.4, 0.15

    def run(jscale=1.0, dh=0.0, ck=0, grads=True):
        lat = _lattice(kind, dims, jscale, dh)
        dJ = np.stack([lat0.bi_J, 0.0 * lat0.bi_J])
        dB = np.stack([np.zeros((N, 3)), np.broadcast_to([0.3, -0.2, 1.0], (N, 3))])
        with GPULattice(lat) as gl:
            gl.set_damping(alpha)
            d = np.einsum("aij,aj->ai", lat.frames, f).reshape(-1)
            gl.set_pulse(np.concatenate([d, d]), amp, 0.1, 3.0, tc, 0.0)
            return AD.adjoint_gradient(gl, init, [[tc, 0.0]] * 2, [[amp, 0.0], [0.0, 0.0]], 0.0, T1, DT, target, W,
                                       dJ if grads else np.zeros((0,)), dB if grads else np.zeros((0,)),
                                       ckpt_interval=ck, want_records=True)

    print(f"[adjoint general] {kind} {dims} alpha {alpha}", flush=True)
    r = run()
    h = 1e-6
    for p, step in enumerate((dict(jscale=1.0), dict(dh=1.0))):
        up = run(**{k: (1.0 if k == "jscale" else 0.0) + h * v for k, v in step.items()}, grads=False)["loss"]
        dn = run(**{k: (1.0 if k == "jscale" else 0.0) - h * v for k, v in step.items()}, grads=False)["loss"]
        fd = (up - dn) / (2.0 * h)
        assert np.all(np.abs(r["grad"][:, p] - fd) <= 1e-6 * np.max(np.abs(r["grad"])))
    for ck in (1, 7, 16):
        c = run(ck=ck)
        assert np.array_equal(c["loss"], r["loss"]) and np.array_equal(c["grad"], r["grad"])
    if kind != "site field":
        o = oracle.OracleLattice(_uc(kind), *dims)
        o.set_alpha(alpha)
        o.set_pulse(f, tc, f * 0.0, 0.0, amp, 0.1, 3.0)
        m = o.integrate_md(init.reshape(-1), 0.0, T1, DT)["mags"].reshape(-1, 9)
        loss = np.sum(W * (m - target) ** 2)
        assert abs(r["loss"][0] - loss) <= 1e-10 * loss
