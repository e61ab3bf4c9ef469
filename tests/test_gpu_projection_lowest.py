"""Entries at and beyond the value with which the projection kernels for K > 8 mark the places that
hold none: in a block whose other entries are feasible they are negative entries like any other."""
import numpy as np
import pytest

from devmem import DeviceArray

pytestmark = pytest.mark.gpu

LOW = {"marker": -1e308, "lowest": -np.finfo(np.float64).max, "minus infinity": -np.inf}


# one K per kernel: 16 lanes a block with 1, 2, 4, 8 values a lane, a wave with 4, 8, 16 and with
# the values in memory; one lane a block with 16, 32, 64 registers and in memory
@pytest.mark.parametrize("K,layout", [(K, 0) for K in (9, 16, 17, 50, 128, 200, 300, 513, 1500)] +
                         [(K, 1) for K in (9, 16, 17, 50, 64, 65, 300)])
@pytest.mark.parametrize("low", sorted(LOW))
def test_lowest_entries_are_projected(ctx, K, layout, low):
    from pasc_inference_amd import capi
    nb = 2 * K + 3
    y = np.zeros((nb, K))
    b = np.arange(nb)
    y[b, b % K] = 1.0               # feasible but for one entry, at every place in turn
    y[b, (b + 1 + b // K) % K] = LOW[low]
    y[-1] = np.eye(K)[0]            # and one feasible block
    host = y.ravel() if layout == 0 else np.ascontiguousarray(y.T).ravel()
    d = DeviceArray(host)
    print(f"lowest entries K={K} layout={layout} {low}", flush=True)
    capi.check(capi.lib().pasc_project_simplex(ctx.h, d.ptr, nb, K, capi.DTYPE_F64, layout, nb))
    out = d.download()
    out = out.reshape(nb, K) if layout == 0 else out.reshape(K, nb).T
    # the threshold of (1, 0, .., 0, low) is 0: the projection is exact
    assert np.array_equal(out, np.where(y > 0.0, y, 0.0))
