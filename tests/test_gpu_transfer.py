"""gamma in and out through the pinned pieces: sizes around the single-thread limit (131072
doubles), one piece (524288) and all of them, both layouts, both storage types, from threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _round_trip(ctx, T, K, prec, seed):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    P = Problem(ctx, np.zeros(T), K, precision=prec)
    g = np.random.default_rng(seed).random((T, K))
    ref = g if prec == 0 else g.astype(np.float32).astype(np.float64)
    for name, a in (("t", g), ("k", g.T)):
        lay = capi.LAYOUT_TMAJOR if name == "t" else capi.LAYOUT_KMAJOR
        P.set_gamma(np.ascontiguousarray(a), lay)
        assert np.array_equal(P.get_gamma(capi.LAYOUT_TMAJOR).reshape(T, K), ref)
        assert np.array_equal(P.get_gamma(capi.LAYOUT_KMAJOR).reshape(K, T), ref.T)
    assert np.array_equal(P.labels(), ref.argmax(1))
    P.set_gamma_uniform()
    u = np.float32(1.0 / K) if prec else 1.0 / K
    assert np.all(P.get_gamma() == u)
    P.close()


@pytest.mark.parametrize("T,K", [(1, 1), (1, 8), (63, 2), (131_072, 1), (131_073, 1), (43_691, 3),
                                 (524_289, 1), (1_398_103, 3), (600_001, 8)])
@pytest.mark.parametrize("prec", [0, 1])
def test_gamma_round_trip(ctx, T, K, prec):
    print(f"T={T} K={K} prec={prec}", flush=True)
    _round_trip(ctx, T, K, prec, T)


def test_gamma_round_trip_from_threads():
    from pasc_inference_amd.solver import Context
    errors = []

    def work(i):
        try:
            with Context(0) as c:
                _round_trip(c, 700_001 + i, 2, i % 2, i)
        except BaseException as e:  # noqa: BLE001 -- reported below
            errors.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors
