"""The flags of the device-driven Krylov solves (csrc/fem_kstate.hpp): no kernel
reads at its entry what one of its own workgroups writes, or its workgroups, and
the wavefronts of one workgroup, would take different ways around a barrier.

The header's functions are what the kernels call; here they run on the host.
Each kernel's entry test is taken before its keeper has written, as by the first
workgroup, and after, as by the last."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COMMON = r"""
#include "fem_kstate.hpp"
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
using namespace femamd;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)
// a kernel: `entry` decides whether a workgroup returns at once, `keeper` is what
// its first workgroup writes
template <class E, class K> bool kernel(KState &st, E entry, K keeper)
{
    const bool first = entry(st);
    keeper(st, first);
    CHECK(entry(st) == first);
    return first;
}
"""

CG = COMMON + r"""
int main()
{
    // residuals 16, 8, 4, ... against tolerance 3 or a limit of steps, in batches
    for (int maxit = 1; maxit < 8; ++maxit)
        for (int look = 0; look < 2; ++look) {
            KState st{};
            st.tol = 3;
            st.maxit = maxit;
            st.res = st.rr = st.n_res = st.n_rr = 16;
            st.fresh = 1;
            int applies = 0;
            for (int step = 0; step < 12; ++step) {
                const double r = 16.0 / (1 << applies);
                kernel(st, cg_skip_dir, [&](KState &s, bool skip) {
                    if (skip) return;
                    const bool stops = cg_stops(s, r, r);
                    cg_keep(s, r, r);
                    CHECK(cg_stops(s, r, r) == stops);   // (every workgroup decides for itself)
                });
                if (!cg_skip_step(st)) ++applies;
                kernel(st, cg_skip_step, [&](KState &s, bool) { cg_pass_on(s); });
                if (look && !cg_skip_dir(st)) {
                    cg_keep(st, 16.0 / (1 << applies), 16.0 / (1 << applies));
                    if (st.end) cg_pass_on(st);
                }
            }
            const int steps = maxit < 3 ? maxit : 3;   // 16 -> 2 takes three
            CHECK(st.done && st.end && applies == steps && st.it == steps && st.res == 16.0 / (1 << steps));
        }
    return 0;
}
"""

GMRES = COMMON + r"""
int main()
{
    // restart m, a limit of steps, residuals 16, 8, 4, ... against tolerance 1 or 0
    for (int m = 1; m < 6; ++m)
        for (int maxit = 1; maxit < 12; ++maxit)
            for (double tol : { 1.5, 0.0 }) {
                KState st{};
                st.gtol = tol;
                st.maxit = maxit;
                int applies = 0, cycles = 0;
                while (!st.converged && st.it < maxit && cycles < 20) {
                    ++cycles;
                    const int before = applies;
                    kernel(st, [](const KState &s) { return gm_skip_scale(s, -1); },
                           [&](KState &s, bool) { gm_begin(s, 16.0 / (1 << applies)); });
                    for (int j = 0; j < m + 2; ++j) {   // (past the end as well)
                        if (!gm_skip_step(st)) ++applies;
                        kernel(st, gm_skip_step, [&](KState &s, bool skip) { if (skip) gm_pass_on(s); });
                        kernel(st, [j](const KState &s) { return gm_skip_scale(s, j); }, [&](KState &s, bool skip) {
                            if (!skip) gm_keep(s, j, m, -16.0 / (1 << applies));
                        });
                    }
                    CHECK(st.jlast == applies - before && st.jlast <= m);
                }
                CHECK(st.it == applies && applies == (maxit < 4 || tol == 0 ? maxit : 4));   // 16 -> 1 takes four
                CHECK(st.converged == (tol > 0 && maxit >= 4));
            }
    return 0;
}
"""


def run(tmp_path, src):
    (tmp_path / "t.cc").write_text(src)
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "dune-fem_amd", "csrc"),
                    str(tmp_path / "t.cc"), "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout


@pytest.mark.parametrize("solver", ["cg", "gmres"])
def test_no_kernel_reads_a_flag_that_it_writes(tmp_path, solver):
    run(tmp_path, {"cg": CG, "gmres": GMRES}[solver])
