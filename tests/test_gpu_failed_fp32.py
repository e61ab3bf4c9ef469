"""An FP32 phase that fails (data whose squares overflow FP32) ends the solve at once, whatever its
iteration cap: the FP64 polish has nothing to run."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_failed_fp32_phase_of_an_image_ends_at_once(ctx):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Problem
    x = 1e25 * np.random.default_rng(0).normal(size=130 * 70)
    P = Problem(ctx, x, 3, T=1, grid_width=130, precision=capi.FP32_BULK, epssqr=2.0)
    P.set_theta(np.array([0.0, 1.0, 3.0]))
    P.set_launch_shape(64, 9, 1)  # the image pass
    took = {}
    for maxit in (100, 100, 200_000):
        print(f"maxit={maxit}", flush=True)
        P.set_gamma_uniform()
        t = time.perf_counter()
        with pytest.raises(capi.PascError) as ei:
            P.gamma_solve(maxit=maxit)
        took[maxit] = time.perf_counter() - t
        assert ei.value.code == 5  # PASC_ERR_NUMERIC
    P.close()
    assert took[200_000] < 0.1 + 2 * took[100]
