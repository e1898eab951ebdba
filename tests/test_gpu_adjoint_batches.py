"""Batches on real adjoint links beyond the lattices whose launches take the
one-wave-per-direction form: packed real links and the 9- and 15-real blocks in the
forms of one thread per (site, right-hand side) and of FP64 lanes, at both storage
precisions and link storages, with one kappa and with one per right-hand side.
"""
import numpy as np
import pytest

from helpers import fold_bc

import leonardym_amd as lym

pytestmark = pytest.mark.gpu

# a last FP64 block of 48 sites in the hop form beside wide batches of the other form, and
# a lattice of which no batched launch takes the hop form (last block of 0 and of 32 sites)
DIMS = [(10, 12, 14, 22), (14, 14, 16, 34)]
EPS = 1e-11   # of the even-odd right-hand side's rule
BOUND = 1e-10  # true residual of the full system, as for the other even-odd solves


def _case(dims, storage):
    ctx = lym.Context(dims, lym.REP_SU2_ADJ)
    U = fold_bc(dims, lym.su2_to_adjoint(lym.gen_su2_links(dims, 0.5, 71)))
    g = lym.Gauge(ctx, U, folded=True, storage=storage)
    V = int(np.prod(dims))
    return ctx, g, [lym.gaussian_spinor(V, 90 + q) for q in range(5)]


def _residual(ctx, g, kappa, x, b):
    out = lym.Spinor(ctx)
    lym.Operator(ctx, lym.OP_CLOVER, 1, kappa, 1.0, False, gauge=g).multiply(out, lym.Spinor(ctx, x))
    return np.linalg.norm((out.download() - b).ravel()) / np.linalg.norm(b.ravel())


@pytest.mark.parametrize("prec", [lym.PREC_SINGLE, lym.PREC_HALF], ids=["fp32", "fp16"])
@pytest.mark.parametrize("storage", [lym.LINKS_FULL, lym.LINKS_RECONSTRUCT], ids=["links9", "links6"])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "x".join(map(str, d)))
def test_widths(dims, storage, prec):
    forms = {w: lym.launch_form(dims, 1, prec, w)["form"] for w in (1, 4)}
    assert forms[4] == lym.FORM_SITE and (forms[1] == lym.FORM_HOP) == (dims == DIMS[0])
    ctx, g, srcs = _case(dims, storage)
    op = lym.Operator(ctx, lym.OP_CLOVER, 1, 0.17, 1.0, True, gauge=g)
    eps = [(EPS * np.linalg.norm(b)) ** 2 for b in srcs]
    got = {}
    for block in (1, 3, 4):
        print("dims", dims, "prec", prec, "block", block, flush=True)
        s = lym.Solver(ctx, lym.SOLVER_PRECOND_MIXED_CG, max_steps=2000, sloppy=prec)
        s.set_rhs_block(block)
        X = [lym.Spinor(ctx) for _ in srcs]
        infos = s.solve_batch(op, [lym.Spinor(ctx, b) for b in srcs], X, eps)
        assert all(i.converged for i in infos)
        got[block] = [x.download() for x in X]
    for q, b in enumerate(srcs):
        assert all(np.array_equal(got[1][q], got[k][q]) for k in (3, 4))
        assert _residual(ctx, g, 0.17, got[4][q], b) <= BOUND


@pytest.mark.parametrize("prec", [lym.PREC_SINGLE, lym.PREC_HALF], ids=["fp32", "fp16"])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "x".join(map(str, d)))
def test_own_kappas(dims, prec):
    ctx, g, srcs = _case(dims, lym.LINKS_FULL)
    op = lym.Operator(ctx, lym.OP_CLOVER, 1, 0.17, 1.0, True, gauge=g)
    kap = [0.15, 0.17, 0.15, 0.165, 0.17]
    eps = [(EPS * np.linalg.norm(b)) ** 2 for b in srcs]

    def run(idx, block):
        print("dims", dims, "prec", prec, "kappas of", idx, flush=True)
        s = lym.Solver(ctx, lym.SOLVER_PRECOND_MIXED_CG, max_steps=2000, sloppy=prec)
        s.set_rhs_block(block)
        X = [lym.Spinor(ctx) for _ in idx]
        infos = s.solve_batch_kappas(op, [kap[q] for q in idx], [lym.Spinor(ctx, srcs[q]) for q in idx], X,
                                     [eps[q] for q in idx])
        assert all(i.converged for i in infos)
        return [x.download() for x in X]

    xs = run(list(range(5)), 4)
    assert np.array_equal(run([3], 1)[0], xs[3])
    for q in range(5):
        assert _residual(ctx, g, kap[q], xs[q], srcs[q]) <= BOUND
