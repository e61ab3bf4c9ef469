"""The kernel-level entry points at the edges of their size rules."""
import numpy as np
import pytest

from devmem import DeviceArray
from helpers import grid_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [9, 15, 17, 32, 33, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2000])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_projection_size_rules(ctx, oracle, K, layout, dtype):
    from pasc_inference_amd import capi
    rng = np.random.default_rng(K)
    nb = 301
    y = rng.normal(size=(nb, K)) * rng.choice([0.05, 1.0, 30.0], size=(nb, 1))
    y[::7] = 1.0 / K                       # ties
    y[3::11] = np.eye(K)[3 % K]            # feasible: left alone
    y[5] = -1e30
    ndt = np.float64 if dtype == "f64" else np.float32
    y = y.astype(ndt).astype(np.float64)
    ref = oracle.project_simplex(y.ravel(), K).reshape(nb, K)
    ld = 0 if layout == 0 else nb + 3      # an odd stride
    host = y.ravel() if layout == 0 else np.pad(y.T, ((0, 0), (0, 3))).ravel()
    d = DeviceArray(host.astype(ndt))
    print(f"projection K={K} layout={layout} {dtype}", flush=True)
    capi.check(capi.lib().pasc_project_simplex(ctx.h, d.ptr, nb, K,
                                               capi.DTYPE_F64 if dtype == "f64" else capi.DTYPE_F32,
                                               layout, ld))
    out = d.download().astype(np.float64)
    out = out.reshape(nb, K) if layout == 0 else out.reshape(K, ld)[:, :nb].T
    # a sum of K terms of size max|y| and one division
    tol = (1e-15 if dtype == "f64" else 1e-7) * K
    scale = np.maximum(1.0, np.abs(y).max(axis=1, keepdims=True))
    keep = np.arange(nb) != 5
    assert np.max((np.abs(out - ref) / scale)[keep]) < tol
    assert out.min() >= 0.0


@pytest.mark.parametrize("K,layout", [(12, 0), (12, 1), (200, 0), (200, 1), (1500, 0)])
def test_projection_of_nonfinite_blocks(ctx, K, layout):
    """NaN takes no part in the search and becomes 0; an infinite entry empties the block."""
    from pasc_inference_amd import capi
    rng = np.random.default_rng(1)
    nb = 70
    y = rng.normal(size=(nb, K))
    clean = y.copy()
    y[10, 4] = np.nan
    y[20] = np.nan
    y[30, 2] = np.inf
    y[40, 5] = -np.inf
    host = y.ravel() if layout == 0 else np.ascontiguousarray(y.T).ravel()
    d = DeviceArray(host)
    capi.check(capi.lib().pasc_project_simplex(ctx.h, d.ptr, nb, K, capi.DTYPE_F64, layout, nb))
    out = d.download()
    out = out.reshape(nb, K) if layout == 0 else out.reshape(K, nb).T
    u = -np.sort(-clean, axis=1)
    h = (np.cumsum(u, 1) - 1.0) / np.arange(1, K + 1)
    tau = h[np.arange(nb), (u > h).sum(1) - 1]
    ref = np.maximum(clean - tau[:, None], 0.0)
    ok = ~np.isin(np.arange(nb), [10, 20, 30, 40])
    assert np.max(np.abs(out - ref)[ok]) < 1e-13
    assert out[10, 4] == 0.0 and abs(out[10].sum() - 1.0) < 1e-12
    assert np.all(out[20] == 0.0) and np.all(out[30] == 0.0)
    assert out[40, 5] == 0.0 and abs(out[40].sum() - 1.0) < 1e-12


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_matvec_size_rules(ctx, oracle, dtype):
    from pasc_inference_amd import capi
    rng = np.random.default_rng(2)
    dt = capi.DTYPE_F64 if dtype == np.float64 else capi.DTYPE_F32
    shapes = [(T, 0, T + o) for T, o in ((1, 0), (2, 1), (63, 0), (64, 1), (65, 3), (255, 0), (256, 1),
                                         (257, 0), (1023, 1), (1024, 0), (1025, 5))]
    shapes += [(w * h, w, w * h + 1) for w, h in ((47, 9), (48, 1), (48, 33), (64, 8), (65, 32),
                                                  (129, 31), (200, 65))]
    for n, w, ld in shapes:
        K, alpha = 3, 0.7
        x = rng.random((K, ld)).astype(dtype)
        dx, dy = DeviceArray(x.ravel()), DeviceArray(np.zeros(K * ld, dtype=dtype))
        T, R = (1, n) if w else (n, 1)
        print(f"matvec n={n} width={w} ld={ld}", flush=True)
        capi.check(capi.lib().pasc_h1_matvec(ctx.h, dx.ptr, dy.ptr, T, R, K, ld, alpha, w, dt))
        out = dy.download().reshape(K, ld)
        xt = np.ascontiguousarray(x[:, :n].T).astype(np.float64).ravel()
        ref = oracle.h1_matvec(xt, T, R, K, alpha, graph=grid_csr(w, n // w) if w else None)
        tol = 1e-14 if dtype == np.float64 else 1e-6
        assert np.max(np.abs(out[:, :n].T - ref.reshape(n, K))) < tol
        assert np.all(out[:, n:] == 0)  # nothing written past the row
