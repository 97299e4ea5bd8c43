"""Dormand-Prince kernel without branches in its right-hand side, where units
of 64 cells are partly empty: one to four sites a thread, and a lattice whose
eleven units do not tile the block (general path).  Same runs and bars as the
full sizes."""
import pytest

from test_gpu_dopri5 import po, test_adaptive_md_vs_oracle as _adaptive  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L1,L2", [(13, 5), (19, 17), (23, 25), (31, 33), (29, 23)])
def test_partly_empty_units(po, L1, L2):  # noqa: F811
    _adaptive(po, L1, L2)
