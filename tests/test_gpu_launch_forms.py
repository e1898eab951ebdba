"""The operators and the FP64 solvers' fused steps against the oracle on lattices whose
launches take each form and block order (checked with lym_launch_form, which makes the
launches' own selection), and the low-precision half-lattice launches at the largest
size of the one-wave-per-direction form.
"""
import numpy as np
import pytest

from helpers import K_CLOVER, K_EO, K_WILSON, OracleField, coords, fold_bc, rel_err_per_site
from test_gpu_launch_shapes import LOWP, neighbour_scale
from test_gpu_parity import Case
from test_launch_form import FP64_FIELD

import leonardym_amd as lym

pytestmark = pytest.mark.gpu

SITE_TOL = 1e-13  # the FP64 apply's bound in every per-site test
SMALL = [f for f in FP64_FIELD if np.prod(f[0]) <= 110000 and f[0] != (14, 14, 14, 14)]


@pytest.mark.parametrize("dims,parity,form,orders", SMALL, ids=lambda v: str(v).replace(", ", "x"))
def test_operators(dims, parity, form, orders):
    assert lym.launch_form(dims, parity)["form"] == form
    print("dims", dims, "parity", parity, "form", form, flush=True)
    case = Case(dims, kappa=0.12, csw=1.0, storage=lym.LINKS_RECONSTRUCT if sum(orders) > 1 else lym.LINKS_FULL)
    psi = case.gauss()
    full = parity < 0 or any(d % 2 for d in dims)
    for kind, okind in (((lym.OP_WILSON, K_WILSON), (lym.OP_CLOVER, K_CLOVER)) if full else ((lym.OP_EO_CLOVER, K_EO),)):
        out = case.spinor(np.full_like(psi, np.nan))
        case.op(kind).multiply(out, case.spinor(psi))
        got, ref = out.download(), case.orc.apply(okind, psi)
        assert np.all(np.isfinite(got)), "sites left unwritten"
        if full:
            assert rel_err_per_site(got, ref) < SITE_TOL
        else:
            odd = coords(dims).sum(1) % 2 == 1
            # two launches and the blocks' inverse (condition below 7 at csw 1)
            assert np.linalg.norm((got - ref)[odd]) < SITE_TOL * np.linalg.norm(ref[odd])


# several site blocks to a sweeping workgroup, so that its sums run over them, and more
# partial sums than a consumer folds by itself (2048)
@pytest.mark.parametrize("method,power", [("cg", 2), ("bicgstab", 1)])
@pytest.mark.parametrize("dims,swept", [((4, 22, 28, 40), True), ((16, 16, 16, 32), True), ((22, 24, 32, 32), False)])
def test_fused_steps(dims, swept, method, power):
    r = lym.launch_form(dims, -1, step=True, part_max=8192)
    assert r["form"] == lym.FORM_STAGED and r["partials"] == r["grid"]
    assert 2 * r["nbpp"] > r["grid"] == 256 if swept else r["partials"] > 2048
    V = int(np.prod(dims))
    U = fold_bc(dims, lym.gen_su3_links(dims, 0.5, 61))
    ctx = lym.Context(dims)
    g = lym.Gauge(ctx, U, folded=True)
    orc = OracleField(dims, U, kappa=0.12, csw=0.0)
    b = lym.gaussian_spinor(V, 62)
    op = lym.Operator(ctx, lym.OP_WILSON, power, 0.12, 0.0, method == "cg", gauge=g)
    for steps in (1, 9) if swept else (2,):
        print("fused", dims, method, steps, flush=True)
        x = lym.Spinor(ctx)
        s = lym.Solver(ctx, lym.SOLVER_CG if method == "cg" else lym.SOLVER_BICGSTAB, precision=1e-30, max_steps=steps)
        info = s.solve(op, lym.Spinor(ctx, b), x)
        ref, _, ok = orc.solve(method, b, 1e-30, max_steps=steps, kind=K_WILSON, power=power, gamma5=method == "cg")
        assert not info.converged and not ok and info.steps == steps
        # sums of 1e7 terms at 1e-16 each, carried over the steps
        assert np.linalg.norm(x.download() - ref) < 1e-11 * np.linalg.norm(ref), steps


@pytest.mark.parametrize("method,kind,power", [("cg", "wilson", 2), ("bicgstab", "clover", 1), ("cg", "eo", 2),
                                               ("bicgstab", "eo", 2)])
@pytest.mark.parametrize("dims", [(6, 4, 4, 6), (12, 12, 12, 24)])
def test_steps_not_fused(dims, method, kind, power, monkeypatch):
    """The iterates where the stencil launches do not take the steps are those where they do
    (rounding of the sums, carried over 9 steps)."""
    V = int(np.prod(dims))
    ctx = lym.Context(dims)
    g = lym.Gauge(ctx, fold_bc(dims, lym.gen_su3_links(dims, 0.5, 61)), folded=True)
    lkind = {"wilson": lym.OP_WILSON, "clover": lym.OP_CLOVER, "eo": lym.OP_EO_CLOVER}[kind]
    op = lym.Operator(ctx, lkind, power, 0.12, 1.0, method == "cg" or power == 2, gauge=g)
    b = lym.Spinor(ctx, lym.gaussian_spinor(V, 62))
    s = lym.Solver(ctx, lym.SOLVER_CG if method == "cg" else lym.SOLVER_BICGSTAB, precision=1e-30, max_steps=9)
    got = []
    for on in ("1", "0", "1"):
        print("steps fused", on, dims, method, kind, flush=True)
        monkeypatch.setenv("LYM_FUSED_FP64", on)
        x = lym.Spinor(ctx)
        assert s.solve(op, b, x).steps == 9
        got.append(x.download())
    assert np.array_equal(got[0], got[2])
    assert np.linalg.norm(got[1] - got[0]) < 1e-11 * np.linalg.norm(got[0])


@pytest.mark.parametrize("prec", [lym.PREC_SINGLE, lym.PREC_HALF], ids=["fp32", "fp16"])
def test_low_precision_half_lattice_at_the_limit(prec):
    dims = (16, 16, 16, 24)
    assert all(lym.launch_form(dims, p, prec, single=True)["form"] == lym.FORM_HOP for p in (0, 1))
    V = int(np.prod(dims))
    ctx = lym.Context(dims)
    g = lym.Gauge(ctx, fold_bc(dims, lym.gen_su3_links(dims, 0.5, 91)), folded=True)
    op = lym.Operator(ctx, lym.OP_EO_CLOVER, 1, 0.13, 1.0, True, gauge=g)
    psi = lym.gaussian_spinor(V, 92)
    ref, got = lym.Spinor(ctx), lym.Spinor(ctx, np.full((V, 4, 3), np.nan + 1j * np.nan))
    op.multiply(ref, lym.Spinor(ctx, psi))
    op.multiply_sloppy(got, lym.Spinor(ctx, psi), prec)
    r, x = ref.download(), got.download()
    assert np.all(np.isfinite(x)), "sites left unwritten"
    s = neighbour_scale(dims, np.linalg.norm(psi.reshape(V, -1), axis=1))
    s = 2 * neighbour_scale(dims, s)  # two hops, through R_ee^-1 (norm below 2)
    err = np.linalg.norm((x - r).reshape(V, -1), axis=1)
    assert np.all(err <= LOWP[prec] * (s + np.linalg.norm(r.reshape(V, -1), axis=1)))
