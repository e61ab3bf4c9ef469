"""The persistent image loop against the image pass (profiling on routes a solve through it) at the
sizes where its tiling can go wrong: one pixel, one column, one row, the edges of a tile's 64 columns
and of its rows for every number of rows per wave (1, 2, 4, 8 by 4 or 8 waves)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(P, g0, profile, **kw):
    P.set_profiling(profile)
    P.set_gamma(g0)
    r = P.gamma_solve(**kw)
    P.set_profiling(False)
    return P.get_gamma(), r


# 65 columns are two tiles: 512 / 1024 / 2048 / 4096 rows are the most that 4 x 1, 8 x 1, 8 x 2 and
# 8 x 4 rows per tile cover with 256 workgroups
@pytest.mark.parametrize("w,h", [(1, 1), (1, 9), (9, 1), (63, 4), (64, 5), (65, 3), (128, 8), (129, 31),
                                 (65, 512), (65, 513), (65, 1031), (65, 2049), (65, 4097), (300, 200)])
@pytest.mark.parametrize("K,prec", [(1, 0), (2, 0), (3, 0), (4, 0), (4, 1), (5, 0), (6, 1), (8, 0), (8, 1)])
def test_image_loop_matches_image_pass(ctx, w, h, K, prec):
    from pasc_inference_amd.solver import Problem, generate_mask
    print(f"{w}x{h} K={K} prec={prec}", flush=True)
    R, xdim = w * h, 1 + K % 3
    rng = np.random.default_rng(100 * w + h)
    theta = rng.random((K, xdim))
    x = theta[rng.integers(0, K, R)] + 0.3 * rng.normal(size=(R, xdim))
    held = generate_mask(3, R, 0.1) if K % 2 == 0 else None
    P = Problem(ctx, x, K, T=1, xdim=xdim, grid_width=w, precision=prec, heldout=held, epssqr=3.0)
    P.set_theta(theta)
    g0 = rng.random(R * K)  # off the simplex
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
    # the residual amplifies gamma by up to 16 epsilon
    assert abs(ra.kkt - rb.kkt) <= 16 * 3.0 * tol


@pytest.mark.parametrize("prec", [0, 1])
def test_image_loop_explicit_term_stops_and_long_runs(ctx, prec):
    """An explicit b, every kind of stop and more iterations than one launch holds, against the
    image pass."""
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    w, h, K = 70, 37, 3
    R = w * h
    rng = np.random.default_rng(5)
    P = Problem(ctx, None, K, T=1, R=R, grid_width=w, precision=prec, epssqr=2.0)
    P.set_linear_term(rng.normal(size=R * K))
    g0 = np.full(R * K, 1.0 / K)
    for kw in (dict(maxit=0), dict(maxit=1), dict(maxit=1000, eps=1e-10),
               dict(maxit=5000, stop_mask=capi.STOP_KKT, kkt_tol=1e-9, kkt_every=4)):
        print(f"prec={prec} {kw}", flush=True)
        ga, ra = _solve(P, g0, True, **kw)
        gb, rb = _solve(P, g0, False, **kw)
        assert (ra.stop_reason, ra.status) == (rb.stop_reason, rb.status)
        assert np.max(np.abs(ga - gb)) <= 1e-5  # two runs stopped by the same test
        assert abs(ra.fx - rb.fx) <= 1e-8 * abs(ra.fx)
    P.close()
