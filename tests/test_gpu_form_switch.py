"""The stencil form of a batch changed on one solver between two calls: each call runs the
form set for it, bit for bit what a fresh solver gives, captured iterations included.
"""
import numpy as np
import pytest

from helpers import fold_bc

import leonardym_amd as lym

pytestmark = pytest.mark.gpu

DIMS = (8, 8, 8, 8)


def _solve(solver, op, srcs, ctx):
    xs = [lym.Spinor(ctx) for _ in srcs]
    infos = solver.solve_batch(op, srcs, xs)
    assert all(i.converged for i in infos)
    return [x.download() for x in xs]


def test_matrix_cores_toggled_on_one_solver():
    ctx = lym.Context(DIMS)
    g = lym.Gauge(ctx, fold_bc(DIMS, lym.gen_su3_links(DIMS, 0.5, 71)), folded=True)
    op = lym.Operator(ctx, lym.OP_CLOVER, 1, 0.13, 1.0, True, gauge=g)
    srcs = [lym.Spinor(ctx, lym.gaussian_spinor(int(np.prod(DIMS)), 80 + q)) for q in range(4)]
    eps = 1e-22 * srcs[0].squared_norm()

    def solver():
        s = lym.Solver(ctx, lym.SOLVER_PRECOND_MIXED_CG, precision=eps, max_steps=2000, sloppy=lym.PREC_HALF)
        s.set_rhs_block(4)
        return s

    fresh = {}
    for mc in (False, True):
        s = solver()
        s.set_matrix_cores(mc)
        fresh[mc] = _solve(s, op, srcs, ctx)
    # the forms differ by rounding, so a replayed capture of the other one shows
    assert not all(np.array_equal(a, b) for a, b in zip(fresh[False], fresh[True]))
    s = solver()
    for mc in (False, True, False, True, True):
        print("matrix cores", mc, flush=True)
        s.set_matrix_cores(mc)
        got = _solve(s, op, srcs, ctx)
        assert s.matrix_cores()[1] == mc
        assert all(np.array_equal(a, b) for a, b in zip(got, fresh[mc])), mc
