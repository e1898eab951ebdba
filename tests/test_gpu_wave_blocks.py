"""FP64 launches in workgroups of one wave (lattices whose site blocks of four waves
would spread badly over the CUs): the operators against the oracle, and the solvers'
fused steps, whose sums have one term a workgroup, against the oracle's iterates.
"""
import numpy as np
import pytest

from helpers import K_CLOVER, K_EO, K_WILSON, coords, rel_err_per_site

import leonardym_amd as lym
from test_gpu_parity import Case

pytestmark = pytest.mark.gpu

# a last block of 16 sites; odd extents; x-slices of whole blocks, and half-lattice
# launches of the form (45000 sites) with a last block of 8
DIMS = [(14, 14, 14, 14), (17, 15, 13, 21), (16, 16, 16, 20), (10, 18, 20, 25), (18, 20, 10, 26)]


@pytest.mark.parametrize("rep", ["su3", "adj"])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "x".join(map(str, d)))
def test_operators(dims, rep):
    even = all(d % 2 == 0 for d in dims)
    case = Case(dims, rep=rep, kappa=0.12, csw=1.0)
    psi = case.gauss()
    for kind, okind in ((lym.OP_WILSON, K_WILSON), (lym.OP_CLOVER, K_CLOVER), (lym.OP_EO_CLOVER, K_EO)):
        if kind == lym.OP_EO_CLOVER and not even:
            continue
        print("dims", dims, rep, "kind", kind, flush=True)
        out = case.spinor(np.full_like(psi, np.nan))
        case.op(kind).multiply(out, case.spinor(psi))
        got, ref = out.download(), case.orc.apply(okind, psi)
        if kind == lym.OP_EO_CLOVER:
            odd = coords(dims).sum(1) % 2 == 1
            # two launches and the blocks' inverse (condition below 7)
            assert np.linalg.norm((got - ref)[odd]) < 1e-13 * np.linalg.norm(ref[odd])
        else:
            assert rel_err_per_site(got, ref) < 5e-14  # 200 roundings of 1.1e-16 at most


@pytest.mark.parametrize("method,kind,power", [("cg", lym.OP_CLOVER, 2), ("bicgstab", lym.OP_WILSON, 1)])
def test_fused_steps(method, kind, power):
    dims = (14, 14, 14, 14)
    case = Case(dims, kappa=0.12, csw=1.0)
    b = case.gauss()
    g5 = method == "cg"
    op = case.op(kind, power=power, gamma5=g5)
    okind = K_CLOVER if kind == lym.OP_CLOVER else K_WILSON
    for steps in (1, 3, 9):
        print("fused", method, steps, flush=True)
        s = lym.Solver(case.ctx, lym.SOLVER_CG if g5 else lym.SOLVER_BICGSTAB, precision=1e-30, max_steps=steps)
        x = case.spinor()
        info = s.solve(op, case.spinor(b), x)
        ref, _, _ = case.orc.solve(method, b, 1e-30, max_steps=steps, kind=okind, power=power, gamma5=g5)
        assert info.steps == steps
        # rounding of the sums (38416 x 24 terms) carried over the steps
        assert np.linalg.norm(x.download() - ref) < 1e-11 * np.linalg.norm(ref), steps
