"""The adjoint of a large problem gives its CG vectors back when it returns, and repeats bit for bit."""
import ctypes as C

import numpy as np
import pytest

from devmem import hip

pytestmark = pytest.mark.gpu


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec", [0, 1])
def test_adjoint_vectors_are_given_back(ctx, prec):
    from pasc_inference_amd.solver import Problem, generate_markov, generate_mask
    T, K = 3_000_000, 8  # six vectors: 1.15 GB
    levels = 1.5 * np.arange(K)
    x, _ = generate_markov(2, T, levels, 1e-3, 0.8)
    mask = generate_mask(3, T, 0.1)
    P = Problem(ctx, x, K, precision=prec, heldout=mask, epssqr=5.0)
    P.set_theta(levels)
    P.gamma_solve(maxit=40, polish_maxit=40, stop_mask=0)
    small = Problem(ctx, x[:5000], K, heldout=mask[:5000], epssqr=5.0)  # the kernels are loaded once
    small.set_theta(levels)
    small.gamma_solve(maxit=40, stop_mask=0)
    small.set_profiling(True)
    small.adjoint(mask[:5000], cg_maxit=20)
    small.close()
    before = _free_bytes()
    out = []
    for _ in range(2):
        print(f"adjoint T={T} prec={prec}", flush=True)
        loss, dle, dth, it = P.adjoint(mask, cg_tol=1e-8, cg_maxit=40)
        out.append(np.concatenate([[loss, dle, it], np.ravel(dth)]))
        assert before - _free_bytes() < 500e6
    P.close()
    assert np.array_equal(out[0], out[1])
