"""A launch shape pinned on a batch of one instance is run, as on a problem: the iterates are those of
the problem with the same pinned shape bit for bit (the persistent loop, which an unpinned
problem of these sizes runs, adds its sums in another order)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KW = dict(maxit=60, polish_maxit=60, stop_mask=0)


def _shape(capi, block, chunk, polish_chunk):
    sh = capi.LaunchShape()
    sh.main = capi.PassShape(block, chunk, 0, 64, 1, 0.0)
    sh.polish = capi.PassShape(block, polish_chunk, 0, 64, 1, 0.0)
    return sh


@pytest.mark.parametrize("prec", [0, 1])
def test_pinned_shape_of_one_series(ctx, prec):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Batch, Problem, generate_markov
    T, levels, eps = 50_001, np.array([0.0, 1.0, 3.0]), 9.0
    x, _ = generate_markov(11, T, levels, 1e-3, 0.8)
    sh = _shape(capi, 128, 4, 2) if prec else _shape(capi, 128, 2, 2)
    print(f"one series prec={prec}", flush=True)
    P = Problem(ctx, x, 3, precision=prec, epssqr=eps)
    P.set_theta(levels)
    P.gamma_solve(**KW)
    loop = P.get_gamma()
    capi.check(capi.lib().pasc_set_launch_shape(P.h, C.byref(sh)))
    P.set_gamma_uniform()
    P.gamma_solve(**KW)
    pinned = P.get_gamma()
    P.close()
    B = Batch(ctx, [x], [3], [levels], [eps], precision=prec)
    capi.check(capi.lib().pasc_batch_set_launch_shape(B.h, C.byref(sh)))
    B.solve(**KW)
    got = B.get_gamma(0, 0)
    B.close()
    assert not np.array_equal(pinned, loop)  # else the comparison below says nothing
    assert np.array_equal(got, pinned)


@pytest.mark.parametrize("prec", [0, 1])
def test_pinned_shape_of_one_image(ctx, prec):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem, ProblemBatch, generate_rect_image
    w, h, K, eps = 130, 70, 3, 2.0
    x, col, _ = generate_rect_image(5, w, h, K, 8, 0.2)
    sh = _shape(capi, 64, 9, 9)
    print(f"one image prec={prec}", flush=True)
    P = Problem(ctx, x, K, T=1, xdim=3, grid_width=w, precision=prec, epssqr=eps)
    P.set_theta(col)
    P.gamma_solve(**KW)
    loop = P.get_gamma()
    capi.check(capi.lib().pasc_set_launch_shape(P.h, C.byref(sh)))
    P.set_gamma_uniform()
    P.gamma_solve(**KW)
    pinned = P.get_gamma()
    P.close()
    B = ProblemBatch(ctx, x, K, col, [eps], precision=prec, T=1, xdim=3, grid_width=w)
    capi.check(capi.lib().pasc_batch_set_launch_shape(B.h, C.byref(sh)))
    B.solve(**KW)
    got = B.get_gamma(0)
    B.close()
    assert not np.array_equal(pinned, loop)
    assert np.array_equal(got, pinned)
