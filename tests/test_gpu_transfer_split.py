"""Transfers at the sizes where their way changes: rows of up to 1 MiB go by the copy engine and are
woven by one thread, larger ones through kernels; host copies of 128 KiB and more (labels of 32768
steps) are shared between threads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = 131_072  # doubles of the padded rows


def _edge(K):
    return ROWS // K // 64 * 64  # the most steps whose rows, padded to 64, are small


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("K,T", [(k, t) for k in range(1, 9) for t in (1, 63, 64, 65, 1001, _edge(k), _edge(k) + 1)])
def test_gamma_both_ways(ctx, K, T, prec):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    print(f"K={K} T={T} prec={prec}", flush=True)
    rng = np.random.default_rng(T + K)
    g = rng.random(T * K)
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


@pytest.mark.parametrize("T", [32_767, 32_768, 32_769, 65_535, 65_536, 65_537, 262_143, 262_145])
def test_labels_where_threads_join(ctx, T):
    from pasc_inference_amd.solver import Problem
    print(f"T={T}", flush=True)
    g = np.random.default_rng(T).random((T, 2))
    P = Problem(ctx, np.zeros(T), 2)
    P.set_theta(np.array([0.0, 1.0]))
    P.set_gamma(g.ravel())
    assert np.array_equal(P.labels(), g.argmax(1))
    P.close()
