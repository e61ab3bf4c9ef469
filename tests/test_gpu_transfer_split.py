"""Transfers at the sizes where the host copy goes from one thread to several (128 KiB, 16384 doubles,
a thread), up and down, in both layouts and both storage types."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("K,n", [(1, 16_383), (1, 16_384), (1, 16_385), (3, 16_383), (1, 32_767), (1, 32_768),
                                 (1, 32_769), (5, 49_155), (1, 131_071), (1, 131_072), (1, 131_073)])
def test_copies_are_whole_where_threads_join(ctx, K, n, prec):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    T = n // K
    assert T * K == n
    print(f"K={K} n={n} prec={prec}", flush=True)
    rng = np.random.default_rng(n)
    g = rng.random(n)
    if prec:
        g = g.astype(np.float32).astype(np.float64)  # what FP32 rows hold
    P = Problem(ctx, rng.random(T), K, precision=prec)
    P.set_theta(np.arange(K, dtype=float))
    P.set_gamma(g)
    up, down = P.get_gamma(), P.get_gamma(capi.LAYOUT_KMAJOR)
    P.set_gamma(down, capi.LAYOUT_KMAJOR)
    again = P.get_gamma()
    P.close()
    assert np.array_equal(up, g) and np.array_equal(again, g)
    assert np.array_equal(down.reshape(K, T), g.reshape(T, K).T)
