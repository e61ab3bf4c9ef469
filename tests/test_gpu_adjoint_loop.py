"""The adjoint's persistent launch against its kernels over device memory (profiling on routes a
call through them) at tile, workgroup and size-rule edges, with more steps than one launch holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEVELS = [0.0, 1.0, 3.0, 4.5, 6.0, 7.5, 9.0, 10.5]


@pytest.mark.parametrize("T", [1, 2, 3, 255, 256, 257, 1023, 1024, 1025, 2049, 262_145, 524_289])
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 8])
def test_adjoint_loop_matches_kernels(ctx, T, K):
    from pasc_inference_amd.solver import Problem, generate_markov, generate_mask
    print(f"T={T} K={K}", flush=True)
    x, _ = generate_markov(T + K, T, LEVELS[:K], 1e-2, 0.8)
    mask = generate_mask(5, T, 0.2)
    P = Problem(ctx, x, K, heldout=mask if K % 2 else None, epssqr=5.0)
    P.set_theta(LEVELS[:K])
    P.gamma_solve(maxit=60, stop_mask=0)
    for kw in (dict(cg_tol=1e-11, cg_maxit=400), dict(cg_tol=1e-30, cg_maxit=3),
               dict(cg_maxit=0)):
        P.set_profiling(True)
        a = P.adjoint(mask, **kw)
        P.set_profiling(False)
        b = P.adjoint(mask, **kw)
        assert a[3] == b[3] or abs(a[3] - b[3]) <= 2  # CG steps (a stop test a rounding away)
        # the same sums in another order (1e-16 a term); lambda to the CG tolerance
        scale = max(1.0, abs(a[1]), np.max(np.abs(a[2])))
        assert abs(a[0] - b[0]) <= 1e-12 * max(1.0, abs(a[0]))
        assert abs(a[1] - b[1]) <= 1e-8 * scale
        assert np.max(np.abs(a[2] - b[2])) <= 1e-8 * scale
    P.close()


def test_adjoint_loop_resumes(ctx):
    """More CG steps than a launch's exchange area holds (512), to the same tolerance."""
    from pasc_inference_amd.solver import Problem, generate_markov, generate_mask
    T, K = 300_000, 3
    x, _ = generate_markov(3, T, LEVELS[:K], 1e-3, 0.8)
    mask = generate_mask(5, T, 0.1)
    P = Problem(ctx, x, K, heldout=mask, epssqr=1000.0)
    P.set_theta(LEVELS[:K])
    P.gamma_solve(maxit=100, stop_mask=0)
    a = P.adjoint(mask, cg_tol=1e-10, cg_maxit=20_000)
    P.set_profiling(True)
    b = P.adjoint(mask, cg_tol=1e-10, cg_maxit=20_000)
    P.close()
    assert a[3] > 512 and abs(a[3] - b[3]) <= 2
    scale = max(1.0, abs(b[1]), np.max(np.abs(b[2])))
    assert abs(a[1] - b[1]) <= 1e-8 * scale
    assert np.max(np.abs(a[2] - b[2])) <= 1e-8 * scale
