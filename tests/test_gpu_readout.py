"""The read-out sums (theta, objective, residual, reconstruction error) against numpy at the edges of
their grid: fewer nodes than a thread pair, a workgroup, the whole grid and one more stride."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,xdim,prec", [(1, 2, 1, 0), (511, 3, 1, 0), (513, 1, 2, 1), (7001, 8, 3, 0),
                                           (524_289, 3, 1, 0), (1_100_003, 4, 1, 1)])
def test_readouts_match_numpy(ctx, T, K, xdim, prec):
    """theta, objective, KKT residual and reconstruction error of a given gamma."""
    from pasc_inference_amd.solver import Problem, generate_mask
    rng = np.random.default_rng(T)
    x = rng.normal(size=(T, xdim))
    held = generate_mask(1, T, 0.3) if T > 1 else None
    g = rng.dirichlet(np.ones(K), size=T)
    if prec:
        g = g.astype(np.float32).astype(np.float64)
    th = rng.normal(size=(K, xdim))
    eps = 2.5
    P = Problem(ctx, x, K, xdim=xdim, precision=prec, heldout=held, epssqr=eps)
    P.set_theta(th)
    P.set_gamma(g)
    obs = np.ones(T, bool) if held is None else held == 0
    q = ((x[:, None, :] - th[None]) ** 2).sum(2) / T * obs[:, None]
    lap = np.zeros_like(g)
    lap[1:] += 2 * (g[1:] - g[:-1])
    lap[:-1] += 2 * (g[:-1] - g[1:])
    grad = eps / T * lap + q
    f = float((0.5 * eps / T * lap * g + q * g).sum())
    z = g - T * grad
    u = -np.sort(-z, axis=1)
    h = (np.cumsum(u, 1) - 1.0) / np.arange(1, K + 1)
    tau = h[np.arange(T), (u > h).sum(1) - 1]
    kkt = np.abs(g - np.maximum(z - tau[:, None], 0)).max()
    fx, kk = P.objective()
    assert abs(fx - f) <= 1e-11 * max(1.0, abs(f)) and abs(kk - kkt) <= 1e-10
    if xdim == 1:
        sol = rng.normal(size=T)
        ref = np.abs(g @ th[:, 0] - sol).sum()
        assert abs(P.abserr(sol) - ref) <= 1e-11 * ref
    got = P.theta_update().reshape(K, xdim)
    s = g[obs].sum(0)
    ref = (g[obs].T @ x[obs]) / s[:, None]
    P.close()
    assert np.max(np.abs(got - ref)) <= 1e-11 * max(1.0, np.abs(ref).max())
