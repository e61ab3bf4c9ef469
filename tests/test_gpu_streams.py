"""Calls on a stream of the caller's leave nothing running on it: the next call may use another."""
import ctypes as C

import numpy as np
import pytest

from devmem import hip

pytestmark = pytest.mark.gpu


class Streams:
    """n streams of the caller's on the context's device."""

    def __init__(self, n):
        self.p = []
        for _ in range(n):
            s = C.c_void_p()
            assert hip().hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
            self.p.append(s)

    def __enter__(self):
        return [s.value for s in self.p]

    def __exit__(self, *a):
        for s in self.p:
            hip().hipStreamDestroy(s)


def idle(stream):
    return hip().hipStreamQuery(C.c_void_p(stream)) == 0


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("T", [5_001, 2_000_003])
def test_explicit_term_set_on_one_stream_and_solved_on_another(prec, T):
    from pasc_inference_amd.solver import Context, Problem
    K = 3
    rng = np.random.default_rng(T)
    bs = [rng.normal(size=T * K) / T for _ in range(3)]
    kw = dict(maxit=6, polish_maxit=4, stop_mask=0)

    def run(streams):
        out = []
        with Context(0) as c:
            P = Problem(c, None, K, T=T, precision=prec, epssqr=2.0)
            for i, b in enumerate(bs):
                if streams:
                    c.set_stream(streams[i % 2])
                P.set_linear_term(b)
                if streams:
                    assert idle(streams[i % 2])
                    c.set_stream(streams[(i + 1) % 2])
                P.set_gamma_uniform()
                r = P.gamma_solve(**kw)
                out.append((P.get_gamma(), r.fx, r.it))
            P.close()
            c.set_stream(None)
        return out

    print(f"explicit term T={T} prec={prec}", flush=True)
    with Streams(2) as s:
        a = run(s)
    for (ga, fa, ia), (gb, fb, ib) in zip(a, run(None)):
        assert np.array_equal(ga, gb) and (fa, ia) == (fb, ib)
