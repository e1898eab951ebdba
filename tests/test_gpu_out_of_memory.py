"""A device allocation that fails in the middle of a solver's setup: the call returns
LYM_ERR_NOMEM and starts nothing, and the next call, with memory there again, sets up
what is missing and gives the solution.

A child process loads a library whose hipMalloc refuses one chosen call, ahead of the
product library; no memory is exhausted.
"""
import os
import subprocess
import sys

import pytest

from helpers import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static int count = 0, refuse = 0;
void shim_refuse(int nth) { count = 0; refuse = nth; }
int shim_count(void) { return count; }
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t) = 0;
    if (!real) {
        void* h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        real = h ? (int (*)(void**, size_t))dlsym(h, "hipMalloc") : 0;
        if (!real) return 999;
    }
    if (++count == refuse) { *p = (void*)0; return 2; }
    return real(p, n);
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
import leonardym_amd as lym

dims = (4, 4, 4, 4)
ctx = lym.Context(dims)
g = lym.Gauge(ctx, lym.gen_su3_links(dims, 0.5, 3), folded=False)
op = lym.Operator(ctx, lym.OP_CLOVER, 1, 0.12, 1.0, True, gauge=g)
b = lym.Spinor(ctx, lym.gaussian_spinor(256, 4))
eps = 1e-22 * b.squared_norm()
checks = {
    "cg": (lym.SOLVER_PRECOND_CG, lambda s, x: [s.solve(op, b, x)]),
    "bicgstab": (lym.SOLVER_PRECOND_BICGSTAB, lambda s, x: [s.solve(op, b, x)]),
    "mixed": (lym.SOLVER_PRECOND_MIXED_CG, lambda s, x: [s.solve(op, b, x)]),
    "batch": (lym.SOLVER_PRECOND_MIXED_CG, lambda s, x: s.solve_batch(op, [b], [x])),
}
for name, (kind, solve) in checks.items():
    def solver():
        s = lym.Solver(ctx, kind, precision=eps, max_steps=2000, sloppy=lym.PREC_HALF)
        s.set_rhs_block(1)
        return s
    x = lym.Spinor(ctx)
    assert all(i.converged for i in solve(solver(), x))  # (the operator's own buffers are there from here on)
    want = x.download()
    shim.shim_refuse(0)
    assert all(i.converged for i in solve(solver(), x))
    n = shim.shim_count()
    assert n > 5, n
    for nth in range(1, n + 1):
        print(name, "refusing allocation", nth, "of", n, flush=True)
        s = solver()
        shim.shim_refuse(nth)
        try:
            solve(s, x)
        except lym.LymError as e:
            assert "bytes" in str(e), e
        else:
            raise AssertionError("the refused allocation went unnoticed")
        shim.shim_refuse(0)
        y = lym.Spinor(ctx)
        assert all(i.converged for i in solve(s, y))
        assert np.array_equal(y.download(), want)
print("ok")
"""


def test_solvers_after_a_refused_allocation(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so), "-ldl"])
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), ROOT], capture_output=True, text=True, timeout=90,
                       env=dict(os.environ))
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok")
