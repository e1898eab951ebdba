"""The FP64 solvers' steps fused into the stencil launches: the iterate after a
given number of steps, on both sides of the chunks of eight steps that are queued
at once, against the oracle's (ConjugateGradient.cpp:10-74,
BiConjugateGradient.cpp:321-507), for launches of both stencil forms.
"""
import numpy as np
import pytest

from helpers import K_CLOVER, K_WILSON, OracleField, fold_bc

import leonardym_amd as lym

pytestmark = pytest.mark.gpu

# the one-wave-per-direction form, the one-thread form with a sweeping grid, and an odd extent
DIMS = [(6, 4, 4, 6), (12, 12, 12, 24), (5, 4, 6, 3)]
STEPS = [1, 2, 8, 9, 17]
# rounding (1e-16 per operation, sums of up to 1e6 terms) grows with the residual's
# recursion over the steps; the iterates compared are far from convergence.  (BiCGStab
# runs on D or Q^2: on the indefinite Q its steps nearly break down, |x| jumps a
# hundredfold, and rounding alone separates two correct iterates by 1e-8 at step 9.)
TOL = 1e-11


@pytest.fixture(scope="module", params=range(len(DIMS)), ids=lambda i: "x".join(map(str, DIMS[i])))
def case(request):
    dims = DIMS[request.param]
    V = int(np.prod(dims))
    U = fold_bc(dims, lym.gen_su3_links(dims, 0.5, 61))
    ctx = lym.Context(dims)
    g = lym.Gauge(ctx, U, folded=True)
    orc = OracleField(dims, U, kappa=0.12, csw=1.0, need_clover=True, need_inverse=False)
    return ctx, g, orc, lym.gaussian_spinor(V, 62)


@pytest.mark.parametrize("method,kind,power", [("cg", "wilson", 2), ("cg", "clover", 2), ("cg", "wilson", 1),
                                               ("bicgstab", "clover", 1), ("bicgstab", "wilson", 2)])
def test_iterates(case, method, kind, power):
    ctx, g, orc, b = case
    okind, lkind = (K_WILSON, lym.OP_WILSON) if kind == "wilson" else (K_CLOVER, lym.OP_CLOVER)
    g5 = method == "cg" or power == 2
    op = lym.Operator(ctx, lkind, power, 0.12, 1.0, g5, gauge=g)
    src, x = lym.Spinor(ctx, b), lym.Spinor(ctx)
    for steps in STEPS if power == 2 or method == "bicgstab" else STEPS[:2]:
        print("dims", ctx.dims, method, kind, power, "steps", steps, flush=True)
        s = lym.Solver(ctx, lym.SOLVER_CG if method == "cg" else lym.SOLVER_BICGSTAB, precision=1e-30,
                       max_steps=steps)
        info = s.solve(op, src, x)
        ref, oinfo, ok = orc.solve(method, b, 1e-30, max_steps=steps, kind=okind, power=power,
                                     gamma5=g5)
        assert not info.converged and not ok and info.steps == steps
        err = np.linalg.norm(x.download() - ref) / np.linalg.norm(ref)
        assert err < TOL, (steps, err)
