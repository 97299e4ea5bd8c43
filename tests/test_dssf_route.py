"""Route of a structure-factor call (csl_dssf_route.hpp), compiled for the
host: the memory that the handle holds from earlier calls does not change it,
and the buffers of the persistent route fit what is available."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = """
#include <cstdio>
#include <cstdlib>
#include "csl_dssf_route.hpp"
int main(int, char** v) {
    auto n = [&](int i) { return size_t(std::strtoull(v[i], nullptr, 10)); };
    const auto r = cslh::dssf_route(n(1), n(2), n(3), n(4), n(5), n(6));
    std::printf("%d %zu\\n", int(r.persistent), r.nc);
}
"""
GB = 1 << 30


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "classical_mcmc_spin_amd", "csrc"),
                    str(d / "t.cpp"), "-o", str(d / "t")], check=True)

    def ask(one_workgroup, n_t, grid, row, free, held):
        out = subprocess.run([str(d / "t"), *map(str, (int(one_workgroup), n_t, grid, row, free, held))], check=True,
                             capture_output=True, text=True).stdout.split()
        return bool(int(out[0])), int(out[1])
    return ask


def sizes(n_t, grid, row, nc):
    return 8 * n_t * grid, 32 * nc * grid, 16 * n_t * row


@pytest.mark.parametrize("A", [1, 2, 16])
@pytest.mark.parametrize("gb", [1, 20, 40, 69, 72])
def test_a_repeated_call_takes_the_same_route(route, A, gb):
    free, n_t = 280 * GB, 1000
    row = gb * GB // (8 * n_t * A)
    first = route(True, n_t, A * row, row, free, 0)
    s, g, q = sizes(n_t, A * row, row, first[1])
    held = (s if first[0] else 0) + g + 2 * q
    if held <= free:
        assert route(True, n_t, A * row, row, free - held, held) == first


@pytest.mark.parametrize("A", [1, 2, 16])
@pytest.mark.parametrize("free_gb", [1, 16, 280])
def test_the_persistent_route_fits(route, A, free_gb):
    n_t, taken = 500, []
    for k in range(1, 40):
        row = free_gb * GB * k // (100 * 8 * n_t * A)
        p, nc = route(True, n_t, A * row, row, free_gb * GB, 0)
        s, g, q = sizes(n_t, A * row, row, nc)
        assert nc >= 1 and nc <= n_t and (nc == 1 or g <= GB // 2)
        if p:
            assert s + g + 2 * q <= 0.75 * free_gb * GB and s <= free_gb * GB / 4
            taken.append(k)
    assert taken == list(range(1, len(taken) + 1)) and taken    # smaller calls fit where larger ones do


def test_larger_lattices_keep_one_sample(route):
    assert route(False, 100, 1000, 500, 100 * GB, 0) == (False, 1)
