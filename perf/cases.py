"""The work that users of this library have it do, as measurable cases.

A case is one call sequence of a user's program through the Python handles (solver.py) or, for
the kernel-level entry points, the C ABI.  `prepare` makes the data and the handle such a program
keeps, `run` is one pass, `exact` restates the pass in plain FP64 torch/numpy.  Every gamma solve
runs a fixed number of SPG iterations (maxit, no early stop) or the reference's own stop at a size
where it comes after a few dozen: the iterates of SPG are sensitive to rounding, and after ~50
iterations two correct orders of summation still agree to 1e-9, after a few hundred they do not.
"""
import ctypes
import math

import numpy as np
import torch

from pasc_inference_amd import capi
from pasc_inference_amd import solver as S

# the launch parameters of a long-running program: host polls every 32 iterations, iterations
# replayed from a HIP graph, the KKT residual on every 4th
TUNED = dict(check_every=32, use_graph=1, kkt_every=4)

LEVELS = [0.0, 1.0, 3.0, 4.5, 6.0, 7.5, 9.0, 10.5]


def listed():
    return [
        # the smallest call: the two-state signal of the parity configuration, the whole
        # theta/gamma alternation with the reference's default stops (launch latency counts)
        dict(name="alternation_1e4", kind="alternation", T=10_000, K=2, eps=10.0, p_switch=0.002,
             sigma=0.5, ts_maxit=4, maxit=40, precision=0),
        # the warm-started epsilon scan of the signal driver (test_signal1D), an odd length
        dict(name="scan_1e5", kind="scan", T=100_003, K=3, eps=30.0, n_eps=3, p_switch=1e-3,
             sigma=1.0, maxit=16, precision=0),
        # the gamma step on a FEM-coarsened time grid (hat functions, a fifth of the steps)
        dict(name="fem_hat_4e5", kind="fem", T=400_001, K=3, eps=30.0, p_switch=1e-3, sigma=0.8,
             reduce=0.2, hat=True, maxit=40, precision=0),
        # the differentiation workload's solve: a tenth of the steps held out, then the read-outs
        # of the result (labels, objective, refitted theta)
        dict(name="heldout_1e6", kind="heldout", T=1_000_000, K=3, eps=30.0, p_switch=1e-3,
             sigma=0.8, frac=0.1, maxit=50, precision=0),
        # the backward direction: gradient of the held-out loss through a converged solve
        dict(name="adjoint_1e6", kind="adjoint", T=1_000_000, K=3, eps=30.0, p_switch=1e-3,
             sigma=0.8, frac=0.1),
        # the alternation on a long series with the FP32 bulk and its FP64 polish
        dict(name="alternation_fp32_3e6", kind="alternation", T=3_000_000, K=3, eps=50.0,
             p_switch=3e-4, sigma=1.0, ts_maxit=2, maxit=12, precision=1),
        # the largest: the headline benchmark's series, FP64
        dict(name="solve_1e7", kind="solve", T=10_000_000, K=3, eps=100.0, p_switch=1e-4,
             sigma=1.0, maxit=50, precision=0),
        # image segmentation: the 1024 x 1024 RGB benchmark image, FP64
        dict(name="image_1024", kind="image", width=1024, height=1024, K=4, xdim=3, eps=10.0,
             maxit=50, precision=0),
        # a small grayscale image of ragged size (the text image of the image driver), FP32 bulk
        dict(name="image_250x150", kind="image", width=250, height=150, K=2, xdim=1, eps=3.0,
             maxit=24, precision=1),
        # the batched epsilon scan of uneven series (FP32 bulk, the batch's default)
        dict(name="batch_8x7", kind="batch", n_series=8, n_eps=7, lg_tmin=4.0, lg_tmax=5.3,
             shape_seed=2, maxit=24, precision=1),
        # a short video: the spatio-temporal graph, 60 frames of 64 x 48
        dict(name="video_60x64x48", kind="video", T=60, width=64, height=48, K=3, eps=5.0,
             maxit=24, precision=0),
        # the kernel-level entry points on the caller's device memory: one projected gradient
        # step x <- P(x - s A x), t-major projection as the reference lays gamma out
        dict(name="kernels_2e6", kind="kernels", T=2_000_003, K=3, dtype="float64", width=0),
    ]


def _log(rng, lo, hi):
    return int(round(10.0 ** rng.uniform(math.log10(lo), math.log10(hi))))


def draw(rng):
    kind = rng.choice(["alternation", "alternation", "scan", "fem", "heldout", "adjoint", "solve",
                       "solve", "image", "image", "batch", "video", "kernels", "kernels"])
    K = rng.choice([2, 2, 3, 3, 4, 5, 8])
    c = dict(kind=kind, K=K, eps=round(10.0 ** rng.uniform(0.7, 2.0), 3),
             p_switch=round(10.0 ** rng.uniform(-4.0, -2.5), 6), sigma=round(rng.uniform(0.4, 1.2), 3))
    if kind == "alternation":
        c.update(T=_log(rng, 2_000, 2_000_000), ts_maxit=rng.choice([2, 3, 4]),
                 precision=rng.choice([0, 1]))
        c.update(maxit=rng.choice([12, 20, 40]) if c["precision"] == 0 else 12)
    elif kind == "scan":
        c.update(T=_log(rng, 2_000, 1_000_000), n_eps=rng.choice([2, 3]), maxit=rng.randint(10, 16),
                 precision=0)
    elif kind == "fem":
        c.update(T=_log(rng, 20_000, 2_000_000), reduce=round(rng.uniform(0.05, 0.7), 3),
                 hat=rng.random() < 0.5, maxit=rng.randint(20, 40), precision=0)
    elif kind == "heldout":
        c.update(T=_log(rng, 5_000, 3_000_000), frac=round(rng.uniform(0.05, 0.3), 3),
                 maxit=rng.randint(25, 50), precision=0)
    elif kind == "adjoint":
        # sizes and smoothing at which the solve converges within prepare's time
        c.update(T=_log(rng, 5_000, 1_000_000), K=rng.choice([2, 3, 4]), frac=0.1, sigma=0.8,
                 eps=round(10.0 ** rng.uniform(0.7, 1.5), 3), p_switch=1e-3)
    elif kind == "solve":
        c.update(T=_log(rng, 2_000, 5_000_000), maxit=rng.randint(25, 50),
                 precision=rng.choice([0, 0, 1]))
        if c["precision"] == 1:
            c["maxit"] = min(c["maxit"], 32)
    elif kind == "image":
        c.update(width=_log(rng, 33, 1100), height=_log(rng, 33, 900), K=rng.choice([2, 3, 4, 5]),
                 xdim=rng.choice([1, 3]), eps=round(10.0 ** rng.uniform(0.0, 1.3), 3),
                 maxit=rng.randint(25, 50), precision=rng.choice([0, 0, 1]))
        if c["precision"] == 1:
            c["maxit"] = min(c["maxit"], 24)
    elif kind == "batch":
        c.update(n_series=rng.randint(3, 8), n_eps=rng.randint(2, 7), lg_tmin=3.5,
                 shape_seed=rng.randint(1, 10_000), lg_tmax=round(rng.uniform(4.5, 5.3), 2),
                 maxit=24, precision=rng.choice([0, 1]))
    elif kind == "video":
        c.update(T=rng.randint(3, 60), width=_log(rng, 9, 70), height=_log(rng, 9, 60),
                 K=rng.choice([2, 3, 4]), eps=round(10.0 ** rng.uniform(0.0, 1.0), 3),
                 maxit=rng.randint(15, 24), precision=0)
    else:
        c.update(K=rng.choice([2, 3, 4, 5, 8, 12, 20, 50]), dtype=rng.choice(["float64", "float32"]),
                 width=rng.choice([0, 0, 1]))
        c.update(T=_log(rng, 5_000, max(20_000, 8_000_000 // c["K"])))
        if c["width"]:
            w = _log(rng, 17, 1000)
            c.update(width=w, T=w * max(1, c["T"] // w))
    return c


# ---- inputs ----------------------------------------------------------------------------------

def _signal(case, seed):
    return S.generate_markov(seed, case["T"], LEVELS[:case["K"]], case["p_switch"], case["sigma"])


def _theta_start(case):
    # fitted levels are near, not at, the true ones
    return np.asarray(LEVELS[:case["K"]]) * 0.95 + 0.1


def _image(case, seed):
    """A rectangle image with xdim channels and its palette [K][xdim]."""
    x, col, _ = S.generate_rect_image(seed, case["width"], case["height"], case["K"], 48, 0.15)
    xd = case["xdim"]
    return (np.ascontiguousarray(x.reshape(-1, 3)[:, :xd]).ravel(),
            np.ascontiguousarray(col.reshape(-1, 3)[:, :xd]).ravel())


def _video(case, seed):
    """[T][R] gray values: a disc moving over a background, with noise."""
    T, w, h = case["T"], case["width"], case["height"]
    rng = np.random.default_rng(seed)
    t, yy, xx = np.meshgrid(np.arange(T), np.arange(h), np.arange(w), indexing="ij")
    cx, cy = w * (0.2 + 0.6 * t / T), h * 0.5
    lab = ((xx - cx) ** 2 + (yy - cy) ** 2 < (0.3 * min(w, h)) ** 2).astype(np.int64)
    lab = np.minimum(lab + 2 * (xx > 0.75 * w), case["K"] - 1)
    return np.asarray(LEVELS)[lab].ravel() + 0.5 * rng.normal(size=T * h * w)


def _eps_list(case):
    return [case["eps"] * 3.0 ** (i - case["n_eps"] + 1) for i in range(case["n_eps"])]


def _batch(case, seed):
    # the lengths and cluster counts belong to the case, the data to the seed
    T, K, lv, p, s, _ = S.generate_batch_params(case["shape_seed"], case["n_series"],
                                                lg_tmin=case["lg_tmin"], lg_tmax=case["lg_tmax"])
    K = [int(k) for k in K]
    th = [np.sort(lv[i, :K[i]]) + 0.3 * np.arange(K[i]) for i in range(len(K))]
    xs = [S.generate_markov(1000 * seed + i, int(T[i]), th[i], float(p[i]), float(s[i]))[0]
          for i in range(len(K))]
    eps = 10.0 ** (-1.0 + 2.5 * np.arange(case["n_eps"]) / max(1, case["n_eps"] - 1))
    return xs, K, th, eps


def _kernel_input(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    K, T = case["K"], case["T"]
    # k-major rows: gamma after a gradient step (most blocks one-hot up to a perturbation)
    lab = torch.randint(0, K, (1, T), generator=g, device="cuda")
    x = torch.zeros((K, T), dtype=torch.float64, device="cuda").scatter_(0, lab, 1.0)
    x += 0.4 * torch.randn((K, T), generator=g, device="cuda", dtype=torch.float64)
    return x.to(getattr(torch, case["dtype"]))


STEP = 0.11  # gradient step of the kernel-level case


class _State:
    pass


def prepare(case, seed):
    st = _State()
    st.case = case
    kind = case["kind"]
    if kind == "kernels":
        st.ctx = S.Context(0)
        st.x = _kernel_input(case, seed)
        st.stream = torch.cuda.Stream()
        st.stream.wait_stream(torch.cuda.current_stream())
        st.ctx.set_stream(st.stream.cuda_stream)
        return st
    st.ctx = S.Context(0)
    K, prec = case.get("K"), case.get("precision", 0)
    if kind in ("alternation", "scan", "solve"):
        st.x, lab = _signal(case, seed)
        st.sol = np.asarray(LEVELS)[lab]
        st.P = S.Problem(st.ctx, st.x, K, precision=prec, epssqr=case["eps"])
    elif kind == "fem":
        st.x, _ = _signal(case, seed)
        st.P = S.Problem(st.ctx, st.x, K, precision=prec, epssqr=case["eps"],
                         fem_reduce=case["reduce"],
                         fem_type=capi.FEM_HAT if case["hat"] else capi.FEM_CONSTANT)
    elif kind in ("heldout", "adjoint"):
        st.x, _ = _signal(case, seed)
        st.mask = S.generate_mask(seed + 1, case["T"], case["frac"])
        st.P = S.Problem(st.ctx, st.x, K, precision=prec, heldout=st.mask, epssqr=case["eps"])
    elif kind == "image":
        st.x, st.theta = _image(case, seed)
        st.P = S.Problem(st.ctx, st.x, K, T=1, xdim=case["xdim"], grid_width=case["width"],
                         precision=prec, epssqr=case["eps"])
    elif kind == "video":
        st.x = _video(case, seed)
        st.P = S.Problem(st.ctx, st.x, K, T=case["T"], grid_width=case["width"], precision=prec,
                         epssqr=case["eps"])
    elif kind == "batch":
        xs, Ks, th, eps = _batch(case, seed)
        st.P = S.Batch(st.ctx, xs, Ks, th, eps, precision=prec)
        st.Ks = Ks
        return st
    if kind != "image":
        st.theta = _theta_start(case) if kind in ("alternation", "scan") else np.asarray(LEVELS[:K])
    st.P.set_theta(st.theta)
    if kind == "adjoint":
        st.P.set_gamma_uniform()
        st.P.gamma_solve(maxit=20_000, stop_mask=capi.STOP_KKT, kkt_tol=1e-12, **TUNED)
    return st


def _spg(case):
    """SPG settings of a fixed budget: maxit iterations, half of them FP64 for the FP32 bulk."""
    n = case["maxit"]
    if case["precision"] == capi.FP32_BULK:
        return dict(maxit=n // 2, polish_maxit=n - n // 2, stop_mask=0, kkt_tol=1e-9)
    return dict(maxit=n, stop_mask=0)


def run(st):
    case, kind = st.case, st.case["kind"]
    if kind == "kernels":
        return _run_kernels(st)
    P = st.P
    if kind == "alternation":
        # TSSolver::solve from uniform gamma and a given start theta, then the result's read-out
        P.set_theta(st.theta)
        P.set_gamma_uniform()
        r = P.ts_solve(ts=dict(maxit=case["ts_maxit"], eps=0.0, skip_first_theta=1), **_spg(case))
        return dict(gamma=P.get_gamma(), theta=P.get_theta(), L=float(r.L), it=int(r.spg_it_sum))
    if kind == "scan":
        P.set_gamma_uniform()
        fx, err = [], []
        for eps in _eps_list(case):
            P.set_epssqr(eps)
            fx.append(float(P.gamma_solve(**_spg(case)).fx))
            err.append(P.abserr(st.sol))
        return dict(gamma=P.get_gamma(), fx=np.asarray(fx), abserr=np.asarray(err))
    if kind in ("solve", "image", "video", "fem"):
        P.set_gamma_uniform()
        more = TUNED if kind == "solve" and case["T"] >= 1_000_000 else {}
        r = P.gamma_solve(**_spg(case), **more)
        return dict(gamma=P.get_gamma(), fx=float(r.fx), it=int(r.it))
    if kind == "heldout":
        P.set_theta(st.theta)
        P.set_gamma_uniform()
        r = P.gamma_solve(**_spg(case), **TUNED)
        f, _ = P.objective()
        return dict(gamma=P.get_gamma(), fx=float(r.fx), objective=f, labels=P.labels(),
                    theta=P.theta_update())
    if kind == "adjoint":
        loss, dle, dth, _ = P.adjoint(st.mask, cg_tol=1e-12, cg_maxit=20_000)
        return dict(loss=loss, dlogeps=dle, dtheta=dth)
    res, _ = P.solve(**_spg(case), **TUNED)
    out = [P.get_gamma(s, e) for s in range(P.n_series) for e in range(P.n_eps)]
    return dict(gamma=out, fx=np.asarray([r.fx for r in res]))


def _run_kernels(st):
    case = st.case
    K, T, w = case["K"], case["T"], case["width"]
    L, h = capi.lib(), st.ctx.h
    dt = capi.DTYPE_F64 if case["dtype"] == "float64" else capi.DTYPE_F32
    with torch.cuda.stream(st.stream):
        y = torch.empty_like(st.x)
        capi.check(L.pasc_h1_matvec(h, ctypes.c_void_p(st.x.data_ptr()),
                                    ctypes.c_void_p(y.data_ptr()), 1 if w else T, T if w else 1, K,
                                    T, 1.0, w, dt))
        z = torch.add(st.x, y, alpha=-STEP)
        zt = z.t().contiguous()  # t-major, K innermost
        capi.check(L.pasc_project_simplex(h, ctypes.c_void_p(zt.data_ptr()), T, K, dt,
                                          capi.LAYOUT_TMAJOR, 0))
        capi.check(L.pasc_project_simplex(h, ctypes.c_void_p(z.data_ptr()), T, K, dt,
                                          capi.LAYOUT_KMAJOR, T))
    return dict(Ax=y, tmajor=zt, kmajor=z)


# ---- the least work of one pass ----------------------------------------------------------------

def _iteration_flops(K, xdim, edges):
    # per node and iteration: the Laplacian, the gradient and data term, the projected step and
    # the natural residual, the three dots and f (edges: graph edges per node)
    return K * (3 * edges + 3 * xdim + 3 + 2 * 6 + 3 * edges + 8) + 8 * K


def work(case):
    kind, K = case["kind"], case["K"] if "K" in case else 3
    if kind == "kernels":
        n, s = case["T"] * K, 8 if case["dtype"] == "float64" else 4
        # x read once; A x, and the two projected layouts written once
        return dict(bytes=4 * n * s, flops=n * (6 if not case["width"] else 10) + 2 * n * 8)
    if kind == "batch":
        T = [10.0 ** ((case["lg_tmin"] + case["lg_tmax"]) / 2)] * case["n_series"]
        n = sum(T)
        return dict(bytes=n * 8 + n * case["n_eps"] * 3 * 8,
                    flops=n * case["n_eps"] * case["maxit"] * _iteration_flops(3, 1, 1))
    if kind == "image":
        n, xd, edges = case["width"] * case["height"], case["xdim"], 2
    elif kind == "video":
        n, xd, edges = case["T"] * case["width"] * case["height"], 1, 7
    else:
        n, xd, edges = case["T"], 1, 1
    if kind == "adjoint":
        # data, mask and gamma in; ~200 CG steps of ~15 flops an entry
        return dict(bytes=n * (8 + 1 + 8 * K), flops=200 * 15 * n * K)
    its = case["maxit"]
    if kind == "alternation":
        its *= case["ts_maxit"]
    elif kind == "scan":
        its *= case["n_eps"]
    nodes = n * case["reduce"] if kind == "fem" else n
    # data in, gamma out, and the arithmetic of the iterations (the iterate can stay on chip)
    return dict(bytes=n * 8 * (xd + K), flops=nodes * its * _iteration_flops(K, xd, edges))


# ---- the same in plain FP64 ------------------------------------------------------------------

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t64(a):
    return torch.as_tensor(np.asarray(a), dtype=torch.float64, device=_dev())


def _tau(y):
    """Threshold of the Euclidean projection of the columns of y [K, n] onto the unit simplex
    (Michelot's support sweeps for few rows, by sorting for many)."""
    K = y.shape[0]
    if K <= 8:
        tau = (y.sum(0) - 1.0) / K
        for _ in range(K - 1):
            on = y > tau
            tau = ((y * on).sum(0) - 1.0) / on.sum(0)
        return tau
    u = torch.sort(y, dim=0, descending=True).values
    h = (torch.cumsum(u, 0) - 1.0) / torch.arange(1, K + 1, dtype=y.dtype, device=y.device)[:, None]
    return torch.gather(h, 0, (u > h).sum(0, keepdim=True) - 1)[0]


def _project(y):
    return torch.clamp(y - _tau(y), min=0.0)


def _lap_time(v):
    a = torch.zeros_like(v)
    d = v[:, 1:] - v[:, :-1]
    a[:, 1:] += 2.0 * d
    a[:, :-1] -= 2.0 * d
    return a


def _spatial_diff(v, u, a):
    """a[.., r] += sum over the 4 neighbours s of (v[.., r] - u[.., s]); [.., h, w]."""
    a[..., 1:, :] += v[..., 1:, :] - u[..., :-1, :]
    a[..., :-1, :] += v[..., :-1, :] - u[..., 1:, :]
    a[..., :, 1:] += v[..., :, 1:] - u[..., :, :-1]
    a[..., :, :-1] += v[..., :, :-1] - u[..., :, 1:]


def _lap_grid(T, h, w):
    def lap(v):
        x = v.view(v.shape[0], T, h, w)
        a = torch.zeros_like(x)
        _spatial_diff(x, x, a)
        if T > 1:
            a[:, 1:] += 2.0 * (x[:, 1:] - x[:, :-1])
            a[:, :-1] += 2.0 * (x[:, :-1] - x[:, 1:])
            _spatial_diff(x[:, 1:], x[:, :-1], a[:, 1:])
            _spatial_diff(x[:, :-1], x[:, 1:], a[:, :-1])
        return a.view_as(v)
    return lap


def _spg_exact(g, q, alpha, lap, maxit, a0=2.0, stop_kkt=0.0, s_kkt=1.0):
    """SPG (m = 20, gamma = 0.9, sigma in [0, 1]) on 1/2 g'(alpha A0)g + <q, g>: the iterate
    after maxit iterations (or at the KKT target), its f and the step of its last direction."""
    g, step, fs, it = _project(g), a0, None, 0
    while True:
        Ag = alpha * lap(g)
        grad = Ag + q
        y = g - step * grad
        tau = _tau(y)
        d = torch.clamp(y - tau, min=0.0) - g
        f = float((0.5 * Ag * g + q * g).sum())
        fs = [f] * 20 if fs is None else fs[1:] + [f]
        if it >= maxit or (stop_kkt and it % 4 == 0 and
                           float((g - _project(g - s_kkt * grad)).abs().max()) <= stop_kkt):
            return g, f, step
        dd, dAd = float((d * d).sum()), float((alpha * lap(d) * d).sum())
        # <grad, d> of a projected step, as a sum of terms of one sign
        gd = -(dd + float((torch.clamp(tau - y, min=0.0) * g).sum())) / step
        if dd == 0.0:
            return g, f, step
        xi, bb = (max(fs) - f) / dAd, -gd / dAd
        beta = min(max(0.9 * bb + math.sqrt(0.81 * bb * bb + 2.0 * xi), 0.0), 1.0)
        g = g + beta * d
        step, it = dd / dAd, it + 1


def _solve_exact(case, g, q, alpha, lap):
    n = case["maxit"]
    if case.get("precision", 0) == capi.FP32_BULK:
        g, _, step = _spg_exact(g, q, alpha, lap, n // 2)
        g, f, _ = _spg_exact(g, q, alpha, lap, n - n // 2, a0=step)
    else:
        g, f, _ = _spg_exact(g, q, alpha, lap, n)
    return g, f


def _data_term(x, theta, scale):
    """[K, n] rows scale * ||x - theta_k||^2; x [n, xdim], theta [K, xdim]."""
    return torch.stack([scale * ((x - th) ** 2).sum(1) for th in theta])


def _uniform(K, n):
    return torch.full((K, n), 1.0 / K, dtype=torch.float64, device=_dev())


def _tmajor(g):
    return g.t().contiguous().view(-1).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "kernels":
        x = _kernel_input(case, seed).double()
        w = case["width"]
        y = (_lap_grid(1, case["T"] // w, w) if w else _lap_time)(x)
        # the step as the caller rounds it in its own type
        z = _project(x - STEP * y)
        return dict(Ax=y, tmajor=z.t().contiguous(), kmajor=z)
    if kind == "batch":
        xs, Ks, th, eps = _batch(case, seed)
        out, fx = [], []
        for x, K, t in zip(xs, Ks, th):
            T = x.size
            q = _data_term(_t64(x)[:, None], _t64(t)[:, None], 1.0 / T)
            for e in eps:
                g, f = _solve_exact(case, _uniform(K, T), q, float(e) / T, _lap_time)
                out.append(_tmajor(g))
                fx.append(f)
        return dict(gamma=out, fx=np.asarray(fx))
    K = case["K"]
    if kind == "image":
        x, theta = _image(case, seed)
        xd, n = case["xdim"], case["width"] * case["height"]
        q = _data_term(_t64(x).view(n, xd), _t64(theta).view(K, xd), 1.0)
        g, f = _solve_exact(case, _uniform(K, n), q, case["eps"],
                            _lap_grid(1, case["height"], case["width"]))
        return dict(gamma=_tmajor(g), fx=f, it=None)
    if kind == "video":
        x, T = _video(case, seed), case["T"]
        q = _data_term(_t64(x)[:, None], _t64(LEVELS[:K])[:, None], 1.0 / T)
        g, f = _solve_exact(case, _uniform(K, x.size), q, case["eps"] / T,
                            _lap_grid(T, case["height"], case["width"]))
        return dict(gamma=_tmajor(g), fx=f, it=None)
    T = case["T"]
    xh, lab = _signal(case, seed)
    x = _t64(xh)[:, None]
    if kind == "alternation":
        th, g = _t64(_theta_start(case))[:, None], _uniform(K, T)
        for i in range(case["ts_maxit"]):
            if i:
                s = g.sum(1)
                th = torch.where(s != 0, (g @ x)[:, 0] / s, torch.zeros_like(s))[:, None]
            g, f = _solve_exact(case, g, _data_term(x, th, 1.0 / T), case["eps"] / T, _lap_time)
        return dict(gamma=_tmajor(g), theta=th[:, 0].cpu().numpy(), L=f, it=None)
    if kind == "scan":
        th, g = _t64(_theta_start(case))[:, None], _uniform(K, T)
        q, sol = _data_term(x, th, 1.0 / T), _t64(np.asarray(LEVELS)[lab])
        fx, err = [], []
        for e in _eps_list(case):
            g, f = _solve_exact(case, g, q, e / T, _lap_time)
            fx.append(f)
            err.append(float(((th * g).sum(0) - sol).abs().sum()))
        return dict(gamma=_tmajor(g), fx=np.asarray(fx), abserr=np.asarray(err))
    th = _t64(LEVELS[:K])[:, None]
    if kind == "solve":
        g, f = _solve_exact(case, _uniform(K, T), _data_term(x, th, 1.0 / T), case["eps"] / T,
                            _lap_time)
        return dict(gamma=_tmajor(g), fx=f, it=None)
    if kind == "fem":
        return _fem_exact(case, x, th)
    held = torch.as_tensor(S.generate_mask(seed + 1, T, case["frac"]) != 0, device=_dev())
    q = _data_term(x, th, 1.0 / T) * (~held)
    if kind == "heldout":
        g, f = _solve_exact(case, _uniform(K, T), q, case["eps"] / T, _lap_time)
        obs = g * (~held)
        s = obs.sum(1)
        return dict(gamma=_tmajor(g), fx=f, objective=f, labels=None,
                    theta=((obs @ x)[:, 0] / s).cpu().numpy())
    return _adjoint_exact(case, x[:, 0], th[:, 0], q, held)


def _fem_exact(case, x, th):
    """Reduce the residual and gamma to the coarse grid, solve there, prolongate (float64)."""
    K, T1 = case["K"], case["T"]
    T2 = math.ceil(T1 * case["reduce"])
    t1 = torch.arange(T1, dtype=torch.float64, device=_dev())
    if case["hat"]:
        diff = (T1 - 1) / (T2 - 1)
        right = math.floor(diff * (T2 - 1))
    else:
        diff = T1 / T2

    def half_up(v):
        return torch.floor(v + 0.5)

    def cells():
        # the constant cell of every fine step
        edges = half_up(torch.arange(T2 + 1, dtype=torch.float64, device=_dev()) * diff)
        return torch.searchsorted(edges, t1, right=True).clamp(1, T2) - 1

    def reduce_(v):
        out = torch.zeros((K, T2), dtype=torch.float64, device=_dev())
        if not case["hat"]:
            return out.index_add_(1, cells(), v)
        span = int(math.ceil(diff)) + 2
        t2 = torch.arange(T2, dtype=torch.float64, device=_dev())
        left, center, rgt = (t2 - 1) * diff, t2 * diff, (t2 + 1) * diff
        start = torch.floor(left)
        for o in range(2 * span + 2):
            t = start + o
            up = t <= center
            phi = torch.where(up, (t - left) / (center - left), (t - rgt) / (center - rgt))
            ok = (t >= 0) & torch.where(up, t < T1, (t < rgt) & (t < right))
            i = t.clamp(0, T1 - 1).long()
            out += torch.where(ok, phi * v[:, i], torch.zeros_like(out))
        return out

    def prolongate(v):
        if not case["hat"]:
            return v[:, cells()]
        tl = torch.floor(t1 / diff)
        a, b = tl * diff, (tl + 1) * diff
        return ((t1 - a) / (b - a) * v[:, (tl + 1).clamp(max=T2 - 1).long()] +
                (t1 - b) / (a - b) * v[:, tl.clamp(max=T2 - 1).long()])

    q = reduce_(_data_term(x, th, 1.0)) / T2
    g, f = _solve_exact(case, reduce_(_uniform(K, T1)), q, case["eps"] / T1, _lap_time)
    return dict(gamma=_tmajor(prolongate(g)), fx=f, it=None)


def _adjoint_exact(case, x, th, q, held):
    """Implicit differentiation of the held-out loss at the minimiser (projected CG, float64)."""
    K, T = case["K"], case["T"]
    alpha = case["eps"] / T
    g, _, _ = _spg_exact(_uniform(K, T), q, alpha, _lap_time, 20_000, stop_kkt=1e-12, s_kkt=T)
    free = g > 1e-12
    nf = free.sum(0)

    def face(v):
        v = torch.where(free, v, torch.zeros_like(v))
        v = torch.where(free, v - v.sum(0) / nf.clamp(min=1), v)
        return torch.where(nf > 1, v, torch.zeros_like(v))

    res = torch.where(held, x - th @ g, torch.zeros_like(x))
    r = face(-2.0 * th[:, None] * res)
    lam, p = torch.zeros_like(r), r.clone()
    rr = rr0 = float((r * r).sum())
    for _ in range(20_000):
        if rr <= 1e-26 * rr0 or rr == 0.0:
            break
        Ap = face(alpha * _lap_time(p))
        pq = float((p * Ap).sum())
        if pq <= 0.0:
            break
        lam += rr / pq * p
        r -= rr / pq * Ap
        new = float((r * r).sum())
        p, rr = r + new / rr * p, new
    dle = -float((lam * alpha * _lap_time(g)).sum())
    dth = (-2.0 * res * g).sum(1) + (lam * 2.0 * (x - th[:, None]) / T * (~held)).sum(1)
    return dict(loss=float((res * res).sum()), dlogeps=dle, dtheta=dth.cpu().numpy())
