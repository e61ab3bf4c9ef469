"""A persistent launch whose workgroups lost each other (here: every launch counts as such) is taken
back: the call goes on in separate launches from where the launch began and gives what those
give by themselves (profiling on), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEVELS = np.array([0.0, 1.0, 3.0])


def _problem(c, kind, prec):
    from pasc_inference_amd.solver import Problem, generate_markov, generate_mask, generate_rect_image
    if kind == "series":
        x, _ = generate_markov(3, 30_001, LEVELS, 1e-3, 0.8)
        P = Problem(c, x, 3, precision=prec, heldout=generate_mask(4, 30_001, 0.1), epssqr=7.0)
        P.set_theta(LEVELS)
    elif kind == "image":
        x, col, _ = generate_rect_image(5, 130, 70, 3, 8, 0.2)
        P = Problem(c, x, 3, T=1, xdim=3, grid_width=130, precision=prec, epssqr=2.0)
        P.set_theta(col)
    else:
        x = np.random.default_rng(6).normal(size=20 * 24 * 20)
        P = Problem(c, x, 3, T=20, grid_width=24, precision=prec, epssqr=2.0)
        P.set_theta(LEVELS)
    return P


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind", ["series", "image", "video"])
def test_lost_launch_is_taken_back(kind, prec):
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Context
    print(f"{kind} prec={prec}", flush=True)
    kw = dict(maxit=30, polish_maxit=20, stop_mask=0)
    with Context(0) as c:
        P = _problem(c, kind, prec)
        g0 = np.random.default_rng(1).random(P.T * P.R * 3)

        def solve():
            P.set_gamma(g0)
            r = P.gamma_solve(**kw)
            return P.get_gamma(), (r.it, r.fx, r.kkt, r.status, r.stop_reason)

        loop = solve()
        P.set_profiling(True)
        passes = solve()
        P.set_profiling(False)
        capi.check(capi.lib().pasc_ctx_set_take_back(c.h, 1))
        lost = [solve(), solve()]
        capi.check(capi.lib().pasc_ctx_set_take_back(c.h, 0))
        again = solve()
        P.close()
    assert not np.array_equal(loop[0], passes[0])  # else the comparison below says nothing
    for got in lost:
        assert np.array_equal(got[0], passes[0]) and got[1] == passes[1]
    assert np.array_equal(again[0], loop[0]) and again[1] == loop[1]


def test_lost_adjoint_is_taken_back():
    from pasc_inference_amd import capi
    from pasc_inference_amd.solver import Context, generate_mask
    mask = generate_mask(4, 30_001, 0.1)
    with Context(0) as c:
        P = _problem(c, "series", 0)
        P.set_gamma_uniform()
        P.gamma_solve(maxit=3000, stop_mask=capi.STOP_KKT, kkt_tol=1e-10)
        out = {}
        for name, on, profile in (("loop", 0, False), ("kernels", 0, True), ("lost", 1, False)):
            print(name, flush=True)
            capi.check(capi.lib().pasc_ctx_set_take_back(c.h, on))
            P.set_profiling(profile)
            loss, dle, dth, it = P.adjoint(mask, cg_tol=1e-10, cg_maxit=2000)
            out[name] = np.concatenate([[loss, dle, it], np.ravel(dth)])
        P.close()
    assert not np.array_equal(out["loop"], out["kernels"])
    assert np.array_equal(out["lost"], out["kernels"])
