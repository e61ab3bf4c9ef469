"""k-major projection of few blocks (a wave a block) and many (a lane a block): both sides of the rule
that takes a call to one or the other, and its time for few large blocks."""
import time

import numpy as np
import pytest

from devmem import DeviceArray

pytestmark = pytest.mark.gpu


def _project(y):
    """The projection of every row (sorted search), row sums in FP64."""
    u = -np.sort(-y, axis=1)
    h = (np.cumsum(u, axis=1) - 1.0) / np.arange(1, y.shape[1] + 1)
    tau = np.take_along_axis(h, (u > h).sum(axis=1, keepdims=True) - 1, axis=1)
    return np.maximum(y - tau, 0.0)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("K,nb", [(33, 1), (33, 5), (33, 8192), (33, 8193), (64, 8193), (65, 3), (65, 131_072),
                                  (65, 131_073), (1024, 7), (1025, 3), (1025, 16_385)])
def test_both_sides_of_the_rule(ctx, K, nb, dtype):
    from pasc_inference_amd import capi
    print(f"k-major K={K} nb={nb} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(K + nb)
    ld = nb + 5
    host = np.full((K, ld), 7.0, dtype=dtype)
    host[:, :nb] = 0.3 * rng.normal(size=(K, nb))
    host[rng.integers(0, K, nb), np.arange(nb)] += 1.0
    d = DeviceArray(host.ravel())
    capi.check(capi.lib().pasc_project_simplex(
        ctx.h, d.ptr, nb, K, capi.DTYPE_F64 if dtype == np.float64 else capi.DTYPE_F32,
        capi.LAYOUT_KMAJOR, ld))
    out = d.download().reshape(K, ld)
    # the last block, the first and a few hundred between
    at = np.unique(np.concatenate([[0, nb - 1], rng.integers(0, nb, 300)]))
    ref = _project(host[:, at].T.astype(np.float64))
    # a sum of K terms of size ~1 and one division, the result rounded to the type
    tol = 1e-15 * K if dtype == np.float64 else 1e-15 * K + 6e-8
    assert np.max(np.abs(out[:, at].T - ref)) < tol
    assert np.all(out[:, nb:] == 7.0)  # nothing beyond the blocks


def test_few_large_blocks_are_not_walked_by_single_lanes(ctx):
    """1000 blocks of 300: k-major takes a few times what t-major takes, not dozens."""
    from pasc_inference_amd import capi
    K, nb = 300, 1000
    y = 0.3 * np.random.default_rng(0).normal(size=K * nb)
    best = {}
    for layout in (capi.LAYOUT_TMAJOR, capi.LAYOUT_KMAJOR):
        d = DeviceArray(y)
        ts = []
        for _ in range(30):
            d.upload(y)
            t = time.perf_counter()
            capi.check(capi.lib().pasc_project_simplex(ctx.h, d.ptr, nb, K, capi.DTYPE_F64, layout, nb))
            ts.append(time.perf_counter() - t)
        best[layout] = min(ts)
    print(f"t-major {best[capi.LAYOUT_TMAJOR] * 1e6:.0f} us, k-major {best[capi.LAYOUT_KMAJOR] * 1e6:.0f} us",
          flush=True)
    assert best[capi.LAYOUT_KMAJOR] < 5 * best[capi.LAYOUT_TMAJOR]
