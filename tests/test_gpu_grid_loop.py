"""The persistent loop of spatio-temporal grids against the graph kernels (profiling on routes a solve
through them) at the sizes where its bricks can go wrong: extents of one, extents that bricks do
not divide, long and flat shapes, and one, two and four nodes per thread."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(P, g0, profile, **kw):
    P.set_profiling(profile)
    P.set_gamma(g0)
    r = P.gamma_solve(**kw)
    P.set_profiling(False)
    return P.get_gamma(), r


@pytest.mark.parametrize("T,w,h", [(2, 1, 1), (2, 5, 1), (3, 1, 7), (7, 13, 11), (4, 211, 3), (301, 5, 4),
                                   (60, 64, 48), (9, 131, 127), (47, 93, 80)])
@pytest.mark.parametrize("K,prec", [(1, 0), (2, 0), (3, 0), (3, 1), (4, 0), (5, 1), (8, 0), (8, 1)])
def test_grid_loop_matches_graph_kernels(ctx, T, w, h, K, prec):
    from pasc_inference_amd.solver import Problem, generate_mask
    print(f"{T} frames {w}x{h} K={K} prec={prec}", flush=True)
    n, xdim = T * w * h, 1 + K % 3
    rng = np.random.default_rng(100 * w + h + T)
    theta = rng.random((K, xdim))
    x = theta[rng.integers(0, K, n)] + 0.3 * rng.normal(size=(n, xdim))
    held = generate_mask(3, n, 0.1) if K % 2 == 0 else None
    P = Problem(ctx, x, K, T=T, xdim=xdim, grid_width=w, precision=prec, heldout=held, epssqr=3.0)
    P.set_theta(theta)
    g0 = rng.random(n * K)  # off the simplex
    # 24 iterations from the same start: two orders of the sums, 1e-16 apart per iteration,
    # agree to 1e-9 (an FP32 phase to the rounding of one FP32 step)
    kw = dict(maxit=24, stop_mask=0) if prec == 0 else dict(maxit=12, polish_maxit=12, stop_mask=0)
    ga, ra = _solve(P, g0, True, **kw)
    gb, rb = _solve(P, g0, False, **kw)
    gc, rc = _solve(P, g0, False, **kw)
    P.close()
    assert (ra.it, ra.stop_reason, ra.status) == (rb.it, rb.stop_reason, rb.status)
    assert np.array_equal(gb, gc) and (rb.fx, rb.kkt) == (rc.fx, rc.kkt)  # repeats bit for bit
    tol = 1e-9 if prec == 0 else 1e-6
    assert np.max(np.abs(ga - gb)) <= tol
    assert abs(ra.fx - rb.fx) <= tol * max(1.0, abs(ra.fx))
    # the residual amplifies gamma by up to 2 x (the weights at a node, 16) epsilon
    assert abs(ra.kkt - rb.kkt) <= 32 * 3.0 * tol


@pytest.mark.parametrize("prec", [0, 1])
def test_grid_loop_explicit_term_stops_and_long_runs(ctx, prec):
    """An explicit b, every kind of stop and more iterations than one launch holds, against the
    graph kernels."""
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    T, w, h, K = 5, 21, 13, 3
    n = T * w * h
    rng = np.random.default_rng(5)
    P = Problem(ctx, None, K, T=T, R=w * h, grid_width=w, precision=prec, epssqr=2.0)
    P.set_linear_term(rng.normal(size=n * K))
    g0 = np.full(n * K, 1.0 / K)
    for kw in (dict(maxit=0), dict(maxit=1), dict(maxit=1000, eps=1e-10),
               dict(maxit=5000, stop_mask=capi.STOP_KKT, kkt_tol=1e-9, kkt_every=4)):
        print(f"prec={prec} {kw}", flush=True)
        ga, ra = _solve(P, g0, True, **kw)
        gb, rb = _solve(P, g0, False, **kw)
        assert (ra.stop_reason, ra.status) == (rb.stop_reason, rb.status)
        assert np.max(np.abs(ga - gb)) <= 1e-5  # two runs stopped by the same test
        assert abs(ra.fx - rb.fx) <= 1e-8 * abs(ra.fx)
    P.close()
