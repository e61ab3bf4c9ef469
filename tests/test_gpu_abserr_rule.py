"""The reconstruction error on both sides of the size from which the solution goes up in shared pieces,
and at the ends of its range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("T", [1, 2, 63, 257, 16_385, 160_000, 160_001, 600_001])
def test_abserr_matches_numpy(ctx, T, prec):
    from pasc_inference_amd.solver import Problem
    print(f"T={T} prec={prec}", flush=True)
    K = 3
    rng = np.random.default_rng(T)
    theta, g, sol = np.array([-1.0, 0.5, 2.0]), rng.random((T, K)), rng.normal(size=T)
    if prec:
        g = g.astype(np.float32).astype(np.float64)  # what FP32 rows hold
    P = Problem(ctx, np.zeros(T), K, precision=prec)
    P.set_theta(theta)
    P.set_gamma(g.ravel())
    got = [P.abserr(sol) for _ in range(2)]
    P.close()
    ref = np.sum(np.abs(g @ theta - sol))
    # T terms of a few roundings each, added in a fixed order
    assert got[0] == got[1] and abs(got[0] - ref) <= 4e-16 * (T + 4) * max(1.0, ref / T)
