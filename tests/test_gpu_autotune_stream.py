"""A batch's autotune that finds its shape in the cache leaves nothing running on a caller's stream."""
import numpy as np
import pytest

from test_gpu_streams import Streams, idle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
def test_cached_batch_autotune_waits_for_its_fill(prec):
    from pasc_inference_amd.solver import Batch, Context, generate_markov
    T, levels = 1_000_003, np.array([0.0, 1.0, 3.0])
    xs = [generate_markov(s, T, levels, 1e-3, 0.8)[0] for s in range(2)]
    eps = list(10.0 ** np.linspace(-1, 1, 12))  # 24 instances: the fill writes 0.3 - 0.6 GB
    print(f"batch autotune prec={prec}", flush=True)
    with Context(0) as c, Streams(2) as s:
        B = Batch(c, xs, [3, 3], [levels, levels], eps, precision=prec)
        c.set_stream(s[0])
        B.autotune()
        for _ in range(5):
            B.autotune()
            assert idle(s[0])
        c.set_stream(s[1])
        res, _ = B.solve(maxit=6, polish_maxit=4, stop_mask=0)
        assert all(r.status == 0 for r in res)
        B.close()
        c.set_stream(None)
