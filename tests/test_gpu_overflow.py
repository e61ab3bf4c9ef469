"""Data whose squares overflow the compute type: the persistent loops of images and videos refuse it
as the passes do (profiling on), in both precisions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("K", [2, 3, 6])
@pytest.mark.parametrize("T,width", [(1, 130), (1, 600), (5, 26)])
def test_overflow_is_refused(ctx, T, width, K, prec):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    n = T * width * 70
    x = (1e25 if prec else 1e170) * np.random.default_rng(K).normal(size=n)
    P = Problem(ctx, x, K, T=T, grid_width=width, precision=prec, epssqr=2.0)
    P.set_theta(np.arange(K, dtype=float))
    for passes in (True, False):
        print(f"T={T} width={width} K={K} prec={prec} passes={passes}", flush=True)
        P.set_profiling(passes)
        P.set_gamma_uniform()
        with pytest.raises(capi.PascError) as ei:
            P.gamma_solve(maxit=30)
        assert ei.value.code == 5  # PASC_ERR_NUMERIC
    P.close()
