"""The persistent 1-D loop against the tiled passes (profiling on routes a solve through them) at
the sizes where its tiling can go wrong: fewer steps than a halo, the edges of a one-wave tile (120
or 248 owned steps), of a workgroup's tiles, and of the chunk and wave rules (1024 tiles)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEVELS = [0.0, 1.0, 3.0, 4.5, 6.0, 7.5, 9.0, 10.5]


def _solve(P, g0, profile, **kw):
    P.set_profiling(profile)
    P.set_gamma(g0)
    r = P.gamma_solve(**kw)
    P.set_profiling(False)
    return P.get_gamma(), r


@pytest.mark.parametrize("T", [1, 2, 3, 5, 119, 120, 121, 247, 248, 249, 479, 480, 481, 993,
                               122_880, 122_881, 253_953, 300_007])
@pytest.mark.parametrize("K,prec", [(1, 0), (2, 0), (3, 0), (4, 1), (5, 0), (8, 1)])
def test_loop_matches_tiled_passes(ctx, T, K, prec):
    from pasc_inference_amd.solver import Problem, generate_markov, generate_mask
    print(f"T={T} K={K} prec={prec}", flush=True)
    x, _ = generate_markov(T + K, T, LEVELS[:K], 1e-2, 0.8)
    held = generate_mask(3, T, 0.1) if K % 2 == 0 else None
    P = Problem(ctx, x, K, precision=prec, heldout=held, epssqr=7.0)
    P.set_theta(LEVELS[:K])
    g0 = np.random.default_rng(T).random(T * K)  # off the simplex
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
    # the residual amplifies gamma by up to 8 epsilon
    assert abs(ra.kkt - rb.kkt) <= 8 * 7.0 * tol


@pytest.mark.parametrize("prec", [0, 1])
def test_loop_explicit_term_stops_and_long_runs(ctx, prec):
    """An explicit b, every kind of stop (iteration cap, |df|, KKT) and more iterations than one
    launch holds, against the tiled passes."""
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    T, K = 3001, 3
    rng = np.random.default_rng(5)
    P = Problem(ctx, None, K, T=T, precision=prec, epssqr=2.0)
    P.set_linear_term(rng.normal(size=T * K) / T)
    g0 = np.full(T * K, 1.0 / K)
    for kw in (dict(maxit=0), dict(maxit=1), dict(maxit=1000, eps=1e-10),
               dict(maxit=5000, stop_mask=capi.STOP_KKT, kkt_tol=1e-9, kkt_every=4)):
        print(f"prec={prec} {kw}", flush=True)
        ga, ra = _solve(P, g0, True, **kw)
        gb, rb = _solve(P, g0, False, **kw)
        assert (ra.stop_reason, ra.status) == (rb.stop_reason, rb.status)
        assert np.max(np.abs(ga - gb)) <= 1e-5  # two runs stopped by the same test
        assert abs(ra.fx - rb.fx) <= 1e-8 * abs(ra.fx)
    if prec == 0:  # (an FP32 phase ends by its own rule at 100 kkt_tol, long before)
        ga, ra = _solve(P, g0, False, maxit=1400, stop_mask=0)
        assert ra.status == 0 and ra.kkt < 1e-7
    P.close()
