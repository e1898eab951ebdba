"""FP64 fields of a batch, one per right-hand side, on lattices whose launches take
the one-thread-per-site stencil (the smaller ones of the other tests take the
one-wave-per-direction form), with a ragged last site block: each solution is the
same bits whatever batch it is solved in, and its residual under the single-field
FP64 operator meets the stopping rule.
"""
import numpy as np
import pytest

from helpers import fold_bc

import leonardym_amd as lym

pytestmark = pytest.mark.gpu

REL = 1e-11
# the stopping rule holds for a recursion-free FP64 residual: what is left between it
# and the one formed here is the rounding of one apply
BOUND = 2e-11


def _case(dims, kappa, power, kind):
    ctx = lym.Context(dims)
    g = lym.Gauge(ctx, fold_bc(dims, lym.gen_su3_links(dims, 0.5, 71)), folded=True)
    V = int(np.prod(dims))
    srcs = [lym.gaussian_spinor(V, 80 + q) for q in range(5)]
    return ctx, g, lym.Operator(ctx, kind, power, kappa, 1.0, power == 2, gauge=g), srcs


def _residual(ctx, op, x, b):
    out = lym.Spinor(ctx)
    op.multiply(out, lym.Spinor(ctx, x))
    return np.linalg.norm((out.download() - b).ravel()) / np.linalg.norm(b.ravel())


@pytest.mark.parametrize("dims,kind,solver,power", [
    ((10, 12, 14, 22), lym.OP_CLOVER, lym.SOLVER_MIXED_CG, 2),
    ((10, 12, 14, 22), lym.OP_WILSON, lym.SOLVER_MIXED_CG, 2),
    ((14, 14, 16, 34), lym.OP_CLOVER, lym.SOLVER_PRECOND_MIXED_CG, 1)])
def test_widths(dims, kind, solver, power):
    ctx, g, op, srcs = _case(dims, 0.11, power, kind)
    eps = [(REL * np.linalg.norm(b)) ** 2 for b in srcs]
    got = {}
    for block in (1, 2, 3, 4, 6):
        print("dims", dims, "block", block, flush=True)
        s = lym.Solver(ctx, solver, max_steps=2000, sloppy=lym.PREC_HALF)
        s.set_rhs_block(block)
        X = [lym.Spinor(ctx) for _ in srcs]
        infos = s.solve_batch(op, [lym.Spinor(ctx, b) for b in srcs], X, eps)
        assert all(i.converged for i in infos)
        got[block] = [x.download() for x in X]
    for q, b in enumerate(srcs):
        assert all(np.array_equal(got[1][q], got[k][q]) for k in (2, 3, 4, 6))
        if solver == lym.SOLVER_MIXED_CG:
            assert _residual(ctx, op, got[4][q], b) <= BOUND
        else:
            assert _residual(ctx, op, got[4][q], b) <= 10 * BOUND  # the rule is on Qhat^2 of the odd half


def test_own_kappas():
    dims = (14, 14, 16, 34)
    ctx, g, op, srcs = _case(dims, 0.11, 1, lym.OP_CLOVER)
    kap = [0.10, 0.11, 0.10, 0.115, 0.11]
    eps = [(REL * np.linalg.norm(b)) ** 2 for b in srcs]

    def run(idx, block):
        print("kappas", idx, "block", block, flush=True)
        s = lym.Solver(ctx, lym.SOLVER_PRECOND_MIXED_CG, max_steps=2000, sloppy=lym.PREC_HALF)
        s.set_rhs_block(block)
        X = [lym.Spinor(ctx) for _ in idx]
        infos = s.solve_batch_kappas(op, [kap[q] for q in idx], [lym.Spinor(ctx, srcs[q]) for q in idx], X,
                                     [eps[q] for q in idx])
        assert all(i.converged for i in infos)
        return [x.download() for x in X]

    xs = run(range(5), 4)
    assert np.array_equal(run([3], 1)[0], xs[3])
    for q in (0, 3):
        o = lym.Operator(ctx, lym.OP_CLOVER, 1, kap[q], 1.0, False, gauge=g)
        assert _residual(ctx, o, xs[q], srcs[q]) <= 10 * BOUND
