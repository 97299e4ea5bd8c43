"""Partitioned kernel with a wave's sites in one sublattice: one to four sites
a thread, parts whose last unit is partly empty, a shape whose waves straddle
two sublattices (the general path), driven and damped.

Bar: 1e-12 against the oracle after 40 RK4 steps: the same FP64 scheme in
another summation order, below 200 roundings of O(1) spins.
"""
import numpy as np
import pytest

from classical_mcmc_spin_amd import GPULattice
from helpers import kitaev, random_state, unit_x_field
from test_gpu_partition import _oracle_refs, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L1,L2,parts,spt,alpha", [
    (13, 7, 1, 1, 0.0),    # a unit of 27 cells
    (31, 33, 1, 2, 0.05),  # sixteen units a sublattice, the last with 63 cells
    (48, 47, 2, 3, 0.0),
    (64, 63, 2, 4, 0.05),
    (40, 40, 2, 2, 0.0),   # thirteen units a sublattice: general path
])
def test_wave_shapes(oracle, L1, L2, parts, spt, alpha):
    uc, lat = kitaev(L1, L2, h=0.1)
    s = random_state(lat, 7)
    f = unit_x_field(lat)
    refs = _oracle_refs(oracle, uc, lat, s, f, 40, alpha=alpha)
    with GPULattice(lat) as gl:
        res = _run(gl, lat, s, f, 40, parts, alpha=alpha)
        assert gl.last_launch_config()["sites_per_thread"] == spt
    for b, ref in enumerate(refs):
        assert np.max(np.abs(res["mags"][:, b] - ref["mags"])) <= 1e-12
        assert np.max(np.abs(res["energy"][:, b] - ref["energy"])) <= 1e-12
        assert np.max(np.abs(res["final"][b] - ref["final"].reshape(-1, 3))) <= 1e-12
