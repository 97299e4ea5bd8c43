"""Plans kept for a shape (csl_plan_pair.hpp), compiled for the host with
plans that record the shape they were made for: after a failure for one shape
(before the first plan, between the two, after both) the next call gets both
plans of the shape it asks for, whichever that is, and no plan leaks."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = """
#include <array>
#include <cstdio>
#include <stdexcept>
#include "csl_plan_pair.hpp"
struct P { int shape; };
static int live = 0;
static void destroy(P* p) { --live; delete p; }
static P* make_one(int shape) { ++live; return new P{shape}; }
using Key = std::array<int, 2>;
int main() {
    int bad = 0;
    for (int fail = 0; fail < 3; ++fail)
        for (int next = 1; next <= 3; ++next) {   // shape asked for after the failure of shape 2
            cslh::PlanPair<P*, Key, destroy> w;
            int made = 0;
            auto ask = [&](int shape, int fail_at) {
                w.use(Key{shape, 1}, [&](P*& a, P*& b) {
                    if (fail_at == 0) throw std::runtime_error("a");
                    a = make_one(shape);
                    if (fail_at == 1) throw std::runtime_error("b");
                    b = make_one(shape);
                    if (fail_at == 2) throw std::runtime_error("c");
                    ++made;
                });
            };
            ask(1, -1);
            ask(1, -1);
            if (made != 1) ++bad, std::printf("plans of a kept shape made again\\n");
            try {
                ask(2, fail);
                ++bad, std::printf("failure swallowed\\n");
            } catch (const std::runtime_error&) {
            }
            if (live != 0) ++bad, std::printf("fail %d: %d plans live after a failure\\n", fail, live);
            ask(next, -1);
            if (!w.a || !w.b || w.a->shape != next || w.b->shape != next)
                ++bad, std::printf("fail %d: shape %d answered by %d %d\\n", fail, next, w.a ? w.a->shape : -1, w.b ? w.b->shape : -1);
        }
    if (live != 0) ++bad, std::printf("%d plans leaked\\n", live);
    return bad != 0;
}
"""


def test_a_failed_shape_leaves_no_plans(tmp_path):
    (tmp_path / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "classical_mcmc_spin_amd", "csrc"),
                    str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
