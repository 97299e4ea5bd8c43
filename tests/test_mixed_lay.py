"""LDS of the mixed lattice's persistent kernel (csl_mixed_lay.hpp), compiled
for the host: every lattice of up to 2048 sites of each species fits a
workgroup, whatever its numbers of sublattices and cells, and the parts of the
layout do not overlap."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = """
#include <cstdio>
#include <initializer_list>
#include "csl_mixed_lay.hpp"
int main() {
    int bad = 0, seen = 0;
    for (int npad = 64; npad <= 2048; npad += 64)
        for (int A2 = 1; A2 * npad <= 2048; ++A2)
            for (int A3 = 1; A3 * npad <= 2048; ++A3)
                for (int nwaves : {8, 16}) {
                    ++seen;
                    const csl::MixPersistLay Y = csl::mix_persist_lay(A2 * npad, A3 * npad, A2, A3, nwaves, false);
                    if (Y.total * 8 > 160 * 1024 && ++bad < 5)
                        std::printf("%d + %d sublattices of %d: %d bytes\\n", A2, A3, npad, Y.total * 8);
                    const int at[] = {Y.t, Y.t2, Y.f, Y.cst, Y.hin, Y.drv, Y.red, Y.total};
                    const int size[] = {6 * A3 * npad + 6, 0, 3 * A2 * npad + 3, Y.tight ? 0 : 3 * Y.rows,
                                        (Y.tight ? 4 : 8) * Y.rows, 24 * Y.chunk, Y.chunk * Y.rec};
                    for (int i = 0; i < 7; ++i)
                        if (at[i] + size[i] > at[i + 1]) ++bad, std::printf("part %d overlaps\\n", i);
                    if (Y.f & 1 || Y.t & 1) ++bad, std::printf("odd offset of a 16-byte record\\n");
                }
    std::printf("%d layouts\\n", seen);
    return bad != 0;
}
"""


def test_every_lattice_of_the_range_fits(tmp_path):
    (tmp_path / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "classical_mcmc_spin_amd", "csrc"),
                    str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
