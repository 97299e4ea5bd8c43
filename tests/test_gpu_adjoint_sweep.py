"""The backward sweep that sums the parameter terms itself, at the edges of its
launch shapes: one to four units of 64 cells a wave, waves with one unit less,
padding lanes, with and without damping, and segments that end inside and at
the ends of the 16-step sums.

Bar: loss and gradient against the FP64 CPU tangent-linear oracle to 1e-10 of
their largest component.  Both integrate the same scheme in FP64; 40 steps of
4 stages leave below 200 roundings of the state and a sum of 160 terms a site,
~1e-13 relative, and the loss gradient cancels at most two to three digits.
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import adjoint as AD
from test_gpu_adjoint import THETA_STAR, W, _oracle_grad, _setup, po  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L1,L2,alpha", [
    (1, 1, 0.02),    # one cell, its bonds to itself
    (8, 8, 0.0),     # exactly one unit a sublattice
    (13, 5, 0.02),   # one cell more than a unit
    (15, 13, 0.02),  # four units, the last with three cells
    (19, 17, 0.0),   # six units on four waves: two and one
    (24, 24, 0.02),  # nine units on four waves: three and two
    (27, 30, 0.02),  # thirteen units, the largest: four and three
    (28, 29, 0.0),
])
def test_sweep_shapes(po, L1, L2, alpha):  # noqa: F811
    n, dt = 40, 0.01
    pulse = (0.5, 0.5, 0.0, 0.2)
    init, T0, T1, target = _setup(po, L1, L2, n, dt, alpha, pulse, seed=L1)
    th = np.stack([THETA_STAR * 1.05, THETA_STAR * 0.93 + 0.01])
    outs = []
    for ck in (0, 16, 7):
        fit = AD.KitaevFit(L1, L2, init, target, T0, T1, dt, pulse=pulse, alpha=alpha, weights=W, ckpt_interval=ck)
        outs.append(fit(th))
        fit.close()
    for lo, g in outs[1:]:
        assert np.array_equal(lo, outs[0][0]) and np.array_equal(g, outs[0][1])
    for b in range(2):
        lo, g = _oracle_grad(po, th[b], L1, L2, init, T0, T1, dt, target, alpha, pulse)
        assert abs(outs[0][0][b] - lo) <= 1e-10 * abs(lo)
        assert np.abs(outs[0][1][b] - g).max() <= 1e-10 * np.abs(g).max()


def test_checkpointed_memory(po):  # noqa: F811
    """With checkpoints a run keeps buffers of one segment: beside the records
    and their loss terms (10 doubles a start and step) and drive factors (6),
    nothing grows with the number of steps but the checkpoints."""
    import torch
    L1, L2, n, dt, ck, B = 6, 6, 4000, 0.002, 64, 64
    pulse = (0.5, 0.5, 0.0, 0.2)
    init, T0, T1, target = _setup(po, L1, L2, n, dt, 0.02, pulse)
    th = np.tile(THETA_STAR * 1.05, (B, 1))
    fit = AD.KitaevFit(L1, L2, init, target, T0, T1, dt, pulse=pulse, alpha=0.02, weights=W, ckpt_interval=ck)
    try:
        torch.cuda.synchronize()
        free0, _ = torch.cuda.mem_get_info()
        fit(th)
        torch.cuda.synchronize()
        free1, _ = torch.cuda.mem_get_info()
    finally:
        fit.close()
    site = 3 * 2 * 64 * 8   # one padded state
    need = B * (ck * 4 * site + (n // ck + 1) * site + n * 16 * 8)
    print(f"[adjoint memory] {(free0 - free1) / 2**20:.0f} MB, buffers that scale {need / 2**20:.0f} MB", flush=True)
    # and under 25 MB of tables, inputs and rounding to pages of 2 MB
    assert free0 - free1 <= need + (25 << 20)
