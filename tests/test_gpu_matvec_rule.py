"""The kernel-level matvec on images on both sides of the rule that takes a call to the image kernel
(0.8 million values over the share of the lanes that have a column), with ragged rows and columns."""
import numpy as np
import pytest

from devmem import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("w,h,K", [(1024, 260, 3), (1024, 261, 3), (1000, 283, 3), (130, 3029, 3), (130, 3030, 3),
                                   (48, 7001, 4), (47, 7001, 4), (1023, 801, 1), (65, 4003, 8)])
def test_image_matvec_on_both_sides(ctx, w, h, K, dtype):
    from pasc_inference_amd import capi
    print(f"matvec {w}x{h} K={K} {dtype.__name__}", flush=True)
    n, ld, alpha = w * h, w * h + 3, 0.7
    x = np.random.default_rng(n).random((K, ld)).astype(dtype)
    dx, dy = DeviceArray(x.ravel()), DeviceArray(np.zeros(K * ld, dtype=dtype))
    capi.check(capi.lib().pasc_h1_matvec(ctx.h, dx.ptr, dy.ptr, 1, n, K, ld, alpha, w,
                                         capi.DTYPE_F64 if dtype == np.float64 else capi.DTYPE_F32))
    out = dy.download().reshape(K, ld)
    v = x[:, :n].astype(np.float64).reshape(K, h, w)
    ref = np.zeros_like(v)
    ref[:, 1:] += v[:, 1:] - v[:, :-1]
    ref[:, :-1] += v[:, :-1] - v[:, 1:]
    ref[:, :, 1:] += v[:, :, 1:] - v[:, :, :-1]
    ref[:, :, :-1] += v[:, :, :-1] - v[:, :, 1:]
    tol = 1e-14 if dtype == np.float64 else 1e-6
    assert np.max(np.abs(out[:, :n] - alpha * ref.reshape(K, n))) < tol
    assert np.all(out[:, n:] == 0)  # nothing written past the row
