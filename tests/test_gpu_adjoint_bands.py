"""The adjoint's CG on images and videos against the same steps in numpy, on both sides of the rule
that gives each XCD a band of nodes (frames of up to 40,960 nodes) and with fewer workgroups than
XCDs.  15 steps from the same right-hand side: two orders of the sums agree to 1e-13 a step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _laplacian(v):
    """A0 v for v [K][T][H][W]: weight 2 to the same pixel of the frames beside, 1 to the four
    neighbours in the frame and in the frames beside."""
    out = np.zeros_like(v)
    T, H, W = v.shape[1:]

    def edge(dt, dy, dx, w):
        a = (slice(None), slice(max(0, -dt), T - max(0, dt)), slice(max(0, -dy), H - max(0, dy)),
             slice(max(0, -dx), W - max(0, dx)))
        b = (slice(None), slice(max(0, dt), T - max(0, -dt)), slice(max(0, dy), H - max(0, -dy)),
             slice(max(0, dx), W - max(0, -dx)))
        out[a] += w * (v[a] - v[b])

    for dt in (-1, 0, 1):
        if abs(dt) >= T:
            continue
        if dt:
            edge(dt, 0, 0, 2.0)
        for dy, dx in ((-1, 0), (1, 0), (0, -1), (0, 1)):
            if abs(dy) < H and abs(dx) < W:
                edge(dt, dy, dx, 1.0)
    return out


@pytest.mark.parametrize("T,w,h,K", [(1, 300, 7, 3), (2, 40, 20, 2), (3, 64, 33, 8), (3, 256, 160, 3),
                                     (3, 241, 170, 3), (1, 700, 300, 4), (9, 101, 97, 5)])
def test_cg_steps_match_numpy(ctx, T, w, h, K):
    from pasc_inference_amd.solver import Problem
    print(f"T={T} {w}x{h} K={K}", flush=True)
    n, eps, steps = T * w * h, 3.0, 15
    rng = np.random.default_rng(n + K)
    theta = 1.5 * np.arange(K)
    x = theta[rng.integers(0, K, n)] + 0.7 * rng.normal(size=n)
    mask = (rng.random(n) < 0.2).astype(np.uint8)
    P = Problem(ctx, x, K, T=T, grid_width=w, heldout=mask, epssqr=eps)
    P.set_theta(theta)
    P.gamma_solve(maxit=6, stop_mask=0)
    g = P.get_gamma().reshape(n, K).T
    loss, dle, dth, it = P.adjoint(mask, cg_tol=1e-14, cg_maxit=steps)
    P.close()

    free = g > 1e-12
    nf = free.sum(0)

    def face(v):
        m = np.where(free, v, 0.0).sum(0) / np.maximum(nf, 1)
        return np.where(free & (nf > 1), v - m, 0.0)

    alpha = eps / n

    def A(v):
        return alpha * _laplacian(v.reshape(K, T, h, w)).reshape(K, n)

    res = np.where(mask == 1, x - theta @ g, 0.0)
    r = face(-2.0 * res * theta[:, None])
    p, lam, rr = r.copy(), np.zeros_like(r), np.sum(r * r)
    for _ in range(steps):
        q = face(A(p))
        pq = np.sum(p * q)
        if not pq > 0.0:
            break
        s = rr / pq
        lam += s * p
        r = r - s * q
        new = np.sum(r * r)
        p, rr = r + new / rr * p, new
    assert it == steps
    ref_loss = np.sum(res * res)
    ref_dle = -np.sum(lam * A(g))
    data = np.where(mask == 1, 0.0, 1.0)
    bscale = -1.0 / n  # b = -(x - theta)^2 / n: its sign cancels below
    ref_dth = -2.0 * (g * res).sum(1) - (lam * 2.0 * (x - theta[:, None]) * data * bscale).sum(1)
    assert abs(loss - ref_loss) <= 1e-10 * ref_loss
    assert abs(dle - ref_dle) <= 1e-8 * np.max(np.abs([ref_dle, ref_loss]))
    assert np.max(np.abs(dth - ref_dth)) <= 1e-8 * max(np.max(np.abs(ref_dth)), ref_loss)
