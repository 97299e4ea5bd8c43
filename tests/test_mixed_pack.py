"""Packed partner tables of the mixed lattice (csl_mixed_pack.hpp), compiled
for the host: an unused slot names what the site's own bonds read anyway (its
matrix is zero, but zero times an infinity or a leftover of unwritten memory is
not), or the record of zeros where it has none, whatever the numbers of
sublattices and cells."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = """
#include <cstdio>
#include <cstdlib>
#include "csl_mixed_pack.hpp"
int main(int argc, char** argv) {
    const int A = std::atoi(argv[1]), Ap = std::atoi(argv[2]), cells = std::atoi(argv[3]), Z = std::atoi(argv[4]);
    const int npad = (cells + 63) / 64 * 64, NP = A * npad;
    // sublattice a has a % (Z + 1) bonds, the k-th to cell (c + k + 1) % cells of sublattice (a + k) % Ap
    std::vector<int> col(size_t(Z) * NP, 0), cnt(NP, 0);
    for (int a = 0; a < A; ++a)
        for (int c = 0; c < cells; ++c) {
            const int p = a * npad + c;
            cnt[p] = a % (Z + 1);
            for (int k = 0; k < cnt[p]; ++k) col[size_t(k) * NP + p] = (a + k) % Ap * npad + (c + k + 1) % cells;
        }
    const auto q = cslh::packed_partners(col.data(), cnt.data(), NP, Z, Ap * npad);
    for (unsigned short v : q) std::printf("%d\\n", int(v));
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("pack")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "classical_mcmc_spin_amd", "csrc"),
                    str(d / "t.cpp"), "-o", str(d / "t")], check=True)
    return str(d / "t")


@pytest.mark.parametrize("A,Ap,cells,Z", [(4, 4, 8, 8), (4, 2, 12, 8), (2, 4, 12, 8), (5, 1, 65, 4), (1, 3, 1, 8),
                                          (4, 2, 64, 4), (6, 3, 100, 4), (32, 1, 60, 8)])
def test_unused_slots(exe, A, Ap, cells, Z):
    out = subprocess.run([exe, *map(str, (A, Ap, cells, Z))], check=True, capture_output=True, text=True).stdout
    npad = (cells + 63) // 64 * 64
    q = np.array(out.split(), dtype=int).reshape(A, npad, Z)
    none = Ap * npad
    assert np.all(q[:, cells:] == none)
    for a in range(A):
        n = a % (Z + 1)
        for k in range(n):
            assert np.array_equal(q[a, :cells, k], (a + k) % Ap * npad + (np.arange(cells) + k + 1) % cells)
        assert np.all(q[a, :cells, n:] == (q[a, :cells, :1] if n else none))
