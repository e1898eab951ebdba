"""BiCGStab's stop with nothing left of the residual: <t, t> == 0 makes the source the
solution (BiConjugateGradient.cpp:449-458), and the whole of it must be copied.
"""
import numpy as np
import pytest

import leonardym_amd as lym

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,kind", [((4, 4, 4, 4), lym.OP_WILSON), ((16, 16, 16, 32), lym.OP_WILSON),
                                       ((5, 4, 6, 3), lym.OP_CLOVER), ((8, 8, 8, 8), lym.OP_EO_CLOVER)])
def test_source_is_the_solution(dims, kind):
    """At kappa = 0 the operator is 1.  Fields of small real integers keep every sum exact
    in any order, so the first step has alpha = 1 and s = t = 0 exactly."""
    V = int(np.prod(dims))
    ctx = lym.Context(dims)
    g = lym.Gauge(ctx, lym.gen_su3_links(dims, 0.5, 3), folded=False)
    op = lym.Operator(ctx, kind, 1, 0.0, 1.0, False, gauge=g)
    r = np.random.default_rng(4)
    b, guess = (r.integers(-3, 4, (V, 4, 3)).astype(complex) for _ in range(2))
    assert np.sum(np.abs(b) ** 2) != np.sum(np.abs(guess) ** 2)
    for _ in range(3):
        print("dims", dims, "kind", kind, flush=True)
        x = lym.Spinor(ctx)
        info = lym.Solver(ctx, lym.SOLVER_BICGSTAB, precision=1e-20, max_steps=50).solve(
            op, lym.Spinor(ctx, b), x, guess=lym.Spinor(ctx, guess))
        assert info.converged and info.steps == 0
        assert np.array_equal(x.download(), b)
