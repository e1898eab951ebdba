"""The stored forms of the clover blocks and their inverses (27 and 36 reals per
chirality on complex links, 9 and 15 on real ones): the FP64 clover operator and the
Schur complement against the oracle, with the unpivoted and the pivoted inverse, and
the low-precision copies against the FP64 operator, from csw = 0 (all numbers of the
stored form are zero) to blocks far from 1, on both stencil forms.
"""
import numpy as np
import pytest

from helpers import K_CLOVER, K_EO, coords, rel_err_per_site

import leonardym_amd as lym
from test_gpu_parity import Case

pytestmark = pytest.mark.gpu

KAPPA = 0.12


@pytest.mark.parametrize("csw", [0.0, 1.0, 6.0])
@pytest.mark.parametrize("rep", ["su3", "adj"])
@pytest.mark.parametrize("dims", [(6, 4, 2, 10), (10, 14, 14, 18)])
def test_operators(dims, rep, csw, monkeypatch):
    case = Case(dims, rep=rep, kappa=KAPPA, csw=csw)
    psi = case.gauss()
    odd = coords(dims).sum(1) % 2 == 1
    norm = np.linalg.norm(psi[odd])
    for pivoted in ("0", "1"):
        monkeypatch.setenv("LYM_CLOVER_INV_PIVOTED", pivoted)
        for kind, okind in ((lym.OP_CLOVER, K_CLOVER), (lym.OP_EO_CLOVER, K_EO)):
            if kind == lym.OP_EO_CLOVER and csw > 1:
                continue  # nothing bounds the blocks' condition there
            print("dims", dims, rep, "csw", csw, "pivoted", pivoted, "kind", kind, flush=True)
            op = case.op(kind)
            out = case.spinor()
            op.multiply(out, case.spinor(psi))
            got, ref = out.download(), case.orc.apply(okind, psi)
            if kind == lym.OP_CLOVER:
                # sums of some 200 products: 200 roundings of 1.1e-16 at most
                assert rel_err_per_site(got, ref) < 5e-14
            # the inverse's error is the rounding times the blocks' condition: six planes with
            # |F| <= 1 each change a block by 6 kappa csw = 0.72 at most at csw 1, so below 7
            assert np.linalg.norm((got - ref)[odd]) < 1e-13 * np.linalg.norm(ref[odd])
            for prec, tol in ((lym.PREC_SINGLE, 2e-6), (lym.PREC_HALF, 4e-3)):
                # FP16 operands carry 2^-11 each (link, spinor, block: 1.5e-3 together,
                # twice through the Schur complement); FP32 2^-24 over some 200 products
                low = case.spinor()
                op.multiply_sloppy(low, case.spinor(psi), prec)
                err = np.linalg.norm((low.download() - got)[odd])
                assert err < tol * max(np.linalg.norm(got[odd]), norm), (prec, err)
