"""The workloads of this framework that its speed is judged by.

A case is one call of a public entry point on a noisy image sequence (blob
phantom drifting by whole pixels, Poisson-Gaussian noise, clipped at 0), or
one training run of the lambda network.  Keys of a sequence case:

  call        how the program calls: "svt" (SVT.denoise on a numpy array),
              "device" (pgsvt_denoise_device on resident frames), "grid"
              (batch.denoise_grid), "learned" (pgsvt_denoise_learned_device)
  n, frames   frame side and sequence length
  dtype       element type of the input
  patch, step, traj      patch size, patch step, trajectory length
  lam         > 0: fixed threshold, no search; 0: chosen by the path
  motion, mwin, median   ARPS on or off, its search window, median radius (0: off)
  expw        exponential weighting (True) or plain soft threshold
  alpha, sigma, mu       noise of the data
  known       the noise parameters are given instead of estimated (the
              estimator needs frames of 2^k pixels a side; given parameters
              allow every size)

"batch" (batch.denoise_batch on sequences of uneven shapes) takes the shapes
of its three jobs from n0, f0, p0, t0, n1, ...; "train" (learned.mlp_train)
rows, n_in, hidden, epochs and batch.
"""

import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pgure-svt_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from pguresvt import SVT, _pguresvt as P, batch, learned  # noqa: E402

_SEQ = dict(call="device", n=256, frames=100, dtype="f32", patch=4, step=1, traj=15, lam=0.0, motion=True, mwin=7,
            median=0, expw=True, alpha=1.0, sigma=8.0, mu=0.0, known=False)
_TORCH = {"u8": torch.uint8, "u16": torch.uint16, "f32": torch.float32, "f64": torch.float64}
_CODE = {"u8": 0, "u16": 1, "f32": 2, "f64": 3}


def _seq(**kw):
    c = dict(_SEQ)
    c.update(kw)
    return c


def listed():
    return [
        # a short clip of a small region at a threshold the user has settled
        # on: the smallest call, where launches and set-up count
        _seq(name="clip_32", call="svt", n=32, frames=16, lam=2.0),
        # the search without motion estimation on a small static sequence
        _seq(name="static_64", call="svt", n=64, frames=20, motion=False, alpha=0.5, sigma=5.0),
        # a detector's 16-bit stack with every default of the estimator
        # (median pre-filter, ARPS, search, noise estimated)
        _seq(name="stack_128_u16", call="svt", n=128, frames=50, dtype="u16", median=5),
        # odd frame side, 8-bit data, a patch and a window outside the
        # instantiated table, plain weighting, noise given
        _seq(name="ragged_99_u8", call="svt", n=99, frames=23, dtype="u8", patch=5, step=2, traj=9, mwin=9, median=2,
             expw=False, alpha=0.8, sigma=4.0, known=True),
        # the same sequence length as the headline at a fixed threshold:
        # reprocessing a resident sequence
        _seq(name="fixed_256", lam=1.0),
        # the headline: lambda searched for every frame of 256 x 256 x 100
        _seq(name="search_256"),
        # a large field of view with a short trajectory, double input
        _seq(name="wide_512_f64", n=512, frames=40, dtype="f64", traj=7),
        # large patches at step 2 on strong noise (the precision study's
        # decomposition, on a field that fits a pass)
        _seq(name="patch8_256", n=256, frames=24, patch=8, step=2, alpha=2.0, sigma=10.0, mu=5.0),
        # the best of 64 lambdas per frame, one sequence
        _seq(name="grid_128", call="grid", n=128, frames=30),
        # uneven sequences in one batch, 64 lambdas per frame
        dict(name="batch_mixed", call="batch", n0=256, f0=30, p0=4, t0=7, n1=128, f1=30, p1=6, t1=15, n2=128, f2=31,
             p2=8, t2=31),
        # lambda proposed by the shipped network, the headline's shape
        _seq(name="learned_256", call="learned"),
        # one training run of the proposal network (its forward and backward)
        dict(name="train_2048", call="train", rows=2048, n_in=3843, hidden=128, epochs=2, batch=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fixed", "fixed", "search", "search", "search", "static", "patch", "grid", "batch", "learned",
                       "train"])
    noise = dict(alpha=round(rng.uniform(0.3, 3.0), 3), sigma=round(rng.uniform(2.0, 15.0), 3))
    if kind == "fixed":
        # any side, every element type, patches of 2 to 4, host or resident
        n, patch = _log_int(rng, 24, 300), rng.choice([2, 3, 4, 4, 4])
        traj = rng.choice([3, 5, 7, 9, 11, 15])
        win = learned.window_length(patch, traj)
        frames = max(win, min(_log_int(rng, 8, 120), int(3e6 / n**2) + 1))
        return _seq(call=rng.choice(["svt", "device"]), n=n, frames=frames, dtype=rng.choice(list(_CODE)), patch=patch,
                    step=rng.choice([1, 1, 2]), traj=traj, lam=round(rng.uniform(0.3, 4.0), 3),
                    median=rng.choice([0, 0, 1, 3, 5]), known=True, expw=rng.random() < 0.8, **noise)
    if kind == "search":
        # estimated noise on sides of 2^k, given noise on any side
        known = rng.random() < 0.5
        n = _log_int(rng, 33, 300) if known else rng.choice([32, 64, 128, 256])
        traj = rng.choice([5, 7, 9, 11, 13, 15])
        frames = max(traj, min(_log_int(rng, 15, 100), int(4e6 / n**2) + 1))
        return _seq(call=rng.choice(["svt", "device"]), n=n, frames=frames, dtype=rng.choice(list(_CODE)),
                    step=rng.choice([1, 1, 1, 2]), traj=traj, median=rng.choice([0, 0, 5]), known=known, **noise)
    if kind == "static":
        n = rng.randint(33, 60)
        traj = rng.choice([5, 9, 15])
        return _seq(call=rng.choice(["svt", "device"]), n=n, frames=rng.randint(traj, 20), traj=traj, motion=False,
                    known=True, dtype=rng.choice(list(_CODE)), **noise)
    if kind == "patch":
        # patches above 4 x 4, from the table and outside it
        patch = rng.choice([5, 6, 7, 8, 8])
        traj = rng.choice([5, 7, 9, 15])
        n, step = _log_int(rng, 48, 200), rng.choice([1, 2, 3])
        frames = max(traj, min(_log_int(rng, 9, 40), int(6e5 * step**2 / n**2) + 1))
        return _seq(call=rng.choice(["svt", "device"]), n=n, frames=frames, dtype=rng.choice(list(_CODE)), patch=patch,
                    step=step, traj=traj, known=True, expw=rng.random() < 0.7, **noise)
    if kind == "grid":
        traj = rng.choice([7, 9, 15])
        n = rng.choice([32, 64, 128])
        return _seq(call="grid", n=n, frames=rng.randint(traj, 40), traj=traj, patch=rng.choice([3, 4, 4, 6]),
                    dtype=rng.choice(list(_CODE)), **noise)
    if kind == "batch":
        c = dict(call="batch")
        for k in range(3):
            n, t = rng.choice([64, 128]), rng.choice([7, 15])
            c.update({"n%d" % k: n, "f%d" % k: rng.randint(t, 30), "p%d" % k: rng.choice([4, 6, 8]), "t%d" % k: t})
        return c
    if kind == "learned":
        n = rng.choice([64, 128, 256])
        return _seq(call="learned", n=n, frames=min(_log_int(rng, 15, 100), int(6e6 / n**2) + 15),
                    dtype=rng.choice(list(_CODE)), **noise)
    return dict(call="train", rows=_log_int(rng, 200, 2048), n_in=256 * rng.choice([3, 7, 15]) + 3, hidden=128,
                epochs=rng.randint(1, 2), batch=rng.choice([64, 128, 256]))


def _frames(n, frames, alpha, sigma, mu, dtype, seed, drift=2, blobs=8):
    """Noisy blob sequence [frames][cols][rows] on the GPU (the column-major
    cube of the C ABI): background 10 plus blobs of sigma 3-8 px and
    amplitude 20-100, each drifting by up to `drift` whole pixels a frame."""
    rng = np.random.Generator(np.random.PCG64(seed))
    cy, cx = rng.uniform(0, n, blobs), rng.uniform(0, n, blobs)
    sig, amp = rng.uniform(3.0, 8.0, blobs), rng.uniform(20.0, 100.0, blobs)
    steps = rng.integers(-drift, drift + 1, size=(frames, blobs, 2)) if drift else np.zeros((frames, blobs, 2))
    steps[0] = 0
    at = np.cumsum(steps, axis=0)
    g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))
    axis = torch.arange(n, dtype=torch.float64, device="cuda")
    ys = torch.from_numpy(cy + at[:, :, 0]).cuda()  # [frames][blobs]
    xs = torch.from_numpy(cx + at[:, :, 1]).cuda()
    w = torch.from_numpy(2.0 * sig**2).cuda()[None, :, None]
    gy = torch.exp(-((axis - ys[:, :, None]) ** 2) / w) * torch.from_numpy(amp).cuda()[None, :, None]
    gx = torch.exp(-((axis - xs[:, :, None]) ** 2) / w)
    clean = 10.0 + (gx[:, :, :, None] * gy[:, :, None, :]).sum(1)
    y = alpha * torch.poisson(clean / alpha, generator=g)
    y += mu + sigma * torch.randn(y.shape, dtype=torch.float64, device="cuda", generator=g)
    y.clamp_(min=0.0)
    if dtype == "u16":  # counts of a 12-bit detector
        return (y * 16).round().clamp_(max=65535).to(torch.int32).to(torch.uint16)
    if dtype == "u8":
        return y.round().clamp_(max=255).to(torch.uint8)
    return y.to(torch.float32).to(_TORCH[dtype])


def _host(cube):
    """numpy (rows, cols, frames), Fortran order."""
    return np.asfortranarray(cube.cpu().numpy().transpose(2, 1, 0))


def _noise_of(c):
    """The (alpha, mu, sigma) handed over where the noise is known, in the
    units of the window normalised to a maximum of 1 (a user's calibration)."""
    if not c["known"]:
        return None, None, None
    return 0.01 * c["alpha"], 0.0, 0.005 * c["sigma"]


def _params(c):
    a, m, s = _noise_of(c)
    return dict(trajectory_length=c["traj"], patch_size=c["patch"], patch_overlap=c["step"], motion_window=c["mwin"],
                motion_filter=c["median"] or -1, noise_method=4, max_iter=500, n_jobs=-1, random_seed=101,
                optimize_pgure=c["lam"] <= 0, exponential_weighting=c["expw"], motion_estimation=c["motion"],
                lambda1=c["lam"] if c["lam"] > 0 else -1.0, noise_alpha=-1.0 if a is None else a,
                noise_mu=-1.0 if m is None else m, noise_sigma=-1.0 if s is None else s, tol=1e-7)


def _bind():
    L = P.load()
    if not getattr(L, "_device_bound", False):
        vp, u32 = C.c_void_p, C.c_uint32
        L.pgsvt_denoise_device.argtypes = [vp, C.c_int, u32, u32, u32, C.POINTER(P.pgsvt_params), vp, vp]
        L.pgsvt_denoise_learned_device.argtypes = [vp, C.c_int, u32, u32, u32, C.POINTER(P.pgsvt_params),
                                                   C.POINTER(learned._Model), vp, vp]
        L._device_bound = True
    return L


_BATCH = dict(learned.TRAIN_PARAMS, random_seed=3)


def prepare(case, seed):
    c, call = case, case["call"]
    if call == "train":
        rng = np.random.Generator(np.random.PCG64(seed))
        X = rng.standard_normal((c["rows"], c["n_in"]), dtype=np.float32)
        t = np.tanh(X[:, :8].sum(1) * 0.5) + 0.1 * rng.standard_normal(c["rows"], dtype=np.float32)
        return dict(call=call, c=c, X=X, t=t.astype(np.float32), p=learned.init_params(c["n_in"], c["hidden"], seed))
    if call == "batch":
        items = []
        for k in range(3):
            n, f, p, t = (c["%s%d" % (q, k)] for q in "nfpt")
            X = _host(_frames(n, f, 1.0, 8.0, 0.0, "f32", 10 * seed + k))
            items.append((X, dict(_BATCH, patch_size=p, trajectory_length=t)))
        return dict(call=call, items=items)
    X = _frames(c["n"], c["frames"], c["alpha"], c["sigma"], c["mu"], c["dtype"], seed, drift=2 if c["motion"] else 0)
    if call == "svt":
        a, m, s = _noise_of(c)
        est = SVT(trajectory_length=c["traj"], patch_size=c["patch"], patch_overlap=c["step"],
                  motion_estimation=c["motion"], motion_window=c["mwin"], motion_filter=c["median"] or None,
                  optimize_pgure=c["lam"] <= 0, lambda1=c["lam"] if c["lam"] > 0 else None,
                  exponential_weighting=c["expw"], noise_alpha=a, noise_mu=m, noise_sigma=s, random_seed=101)
        return dict(call=call, X=_host(X), svt=est)
    if call == "grid":
        return dict(call=call, X=_host(X), params=_params(c))
    s = dict(call=call, c=c, X=X, p=P.make_params(**_params(c)), lib=_bind(),
             Y=torch.empty(X.shape, dtype=torch.float64, device="cuda"),
             est=np.empty((4, c["frames"])))
    if call == "learned":
        s["model"] = learned.LambdaModel.load(learned.default_model_path())
        s["model_c"] = s["model"]._c()
    torch.cuda.synchronize()  # the library works on a stream of its own
    return s


def run(state):
    call = state["call"]
    if call == "svt":
        r = state["svt"].denoise(state["X"])
        return dict(Y=r.Y_, lambdas=r.lambda1s_, alphas=r.noise_alphas_, mus=r.noise_mus_, sigmas=r.noise_sigmas_)
    if call == "grid":
        Y, est = batch.denoise_grid(state["X"], n_lambda=64, **state["params"])
        return dict(Y=Y, estimates=est)
    if call == "batch":
        outs = batch.denoise_batch(state["items"], n_lambda=64, concurrency=4)
        return [dict(Y=Y, estimates=est) for Y, est in outs]
    if call == "train":
        c = state["c"]
        p, losses = learned.mlp_train(state["X"], state["t"], state["p"], c["epochs"], c["batch"], 1e-3, 0, c["hidden"])
        return dict(params=p, losses=losses)
    c, lib, X, Y, est = state["c"], state["lib"], state["X"], state["Y"], state["est"]
    head = (X.data_ptr(), _CODE[c["dtype"]], c["n"], c["n"], c["frames"], C.byref(state["p"]))
    tail = (Y.data_ptr(), est.ctypes.data)
    if call == "learned":
        P.check(lib.pgsvt_denoise_learned_device(*head, C.byref(state["model_c"]), *tail))
    else:
        P.check(lib.pgsvt_denoise_device(*head, *tail))
    return dict(Y=Y, estimates=est)


def _window_work(n, frames, patch, step, traj, variants, evals):
    """Bytes and operations of a sequence: thin SVDs (14 m n^2 + 8 n^3 each),
    threshold and reconstruction of every patch per evaluated lambda."""
    nw, m = learned.window_length(patch, traj), patch * patch
    side = len(set(range(0, n - patch + 1, step)) | {n - patch})
    mats = float(side * side * frames)
    return mats * variants * (14 * m * nw**2 + 8 * nw**3) + mats * evals * (2 * m * nw + 3 * m)


# lambda evaluations per window: the search stops after about 19 distinct
# ones at tol 1e-7 (the learned path's probe needs at least three)
_SEARCH, _PROBE, _GRID = 19, 3, 64


def work(case):
    c, call = case, case["call"]
    if call == "train":
        h, k = c["hidden"], c["n_in"]
        macs = c["rows"] * (k * h + 2 * h * h + h)
        weights = learned.param_count(k, h)
        return {"bytes": 4.0 * (c["rows"] * (k + 1) + 2 * weights), "flops": 6.0 * c["epochs"] * macs}
    if call == "batch":
        b = f = 0.0
        for k in range(3):
            n, fr, p, t = (c["%s%d" % (q, k)] for q in "nfpt")
            b += 12.0 * n * n * fr
            f += _window_work(n, fr, p, 1, t, 3, _GRID)
        return {"bytes": b, "flops": f}
    cells = float(c["n"] ** 2 * c["frames"])
    size = {"u8": 1, "u16": 2, "f32": 4, "f64": 8}[c["dtype"]]
    if call == "learned":
        variants, evals = 1, _PROBE
    elif call == "grid":
        variants, evals = 3, _GRID
    else:
        variants, evals = (1, 1) if c["lam"] > 0 else (3, _SEARCH)
    return {"bytes": cells * (size + 8), "flops": _window_work(c["n"], c["frames"], c["patch"], c["step"], c["traj"],
                                                              variants, evals)}


# ------------------------------------------------------------------ exact --
def _block_cost(S, F, i, j, r, c, bs):
    """Mean squared difference of the bs x bs blocks of S at (i, j) and of F
    at (r, c), for vectors of positions (frames indexed [col][row])."""
    cost = torch.zeros(i.shape, dtype=torch.float64, device=S.device)
    for q in range(bs * bs):
        d = S[j + q // bs, i + q % bs] - F[c + q // bs, r + q % bs]
        cost += d * d
    return cost / (bs * bs)


def _arps(S, F, i, j, pm, mw, bs):
    """Adaptive rood pattern search of every block of S in F: the large
    pattern (step from the predicted motion pm, or 2 in the first column),
    then the small one until its centre is the best; offsets already looked
    at are skipped, ties go to the first point."""
    n = S.shape[0] - bs
    w = 2 * mw + 1
    dev, cnt = S.device, i.numel()
    far = torch.full((cnt,), 1e9, dtype=torch.float64, device=dev)
    rows = torch.arange(cnt, device=dev)
    seen = torch.zeros((cnt, w * w), dtype=torch.bool, device=dev)

    def look(r, c, skip):
        cost = _block_cost(S, F, i, j, r.clamp(0, n), c.clamp(0, n), bs)
        return torch.where(skip, far, cost)

    def mark(r, c, ok):
        ok = ok & (r >= 0) & (r < w) & (c >= 0) & (c < w)
        at = (r + w * c).clamp(0, w * w - 1)
        seen[rows[ok], at[ok]] = True

    cost = _block_cost(S, F, i, j, i, j, bs)
    zero = torch.zeros_like(i)
    mark(zero + mw, zero + mw, zero == 0)
    py, px = pm
    ay, ax = py.abs(), px.abs()
    step = torch.maximum(ay, ax)
    rood = ((ay == 0) & (ax == step)) | ((ax == 0) & (ay == step))
    first = j == 0
    step = torch.where(first, 2, step)
    points = torch.where(first | rood, 5, 6)
    best, by, bx = None, None, None
    for k, (v, h) in enumerate([(-step, zero), (zero, -step), (zero, zero), (zero, step), (step, zero), (py, px)]):
        if k == 2:
            ck = cost
        else:
            r, c = i + v, j + h
            skip = (step == 0) | (r < 0) | (c < 0) | (r > n) | (c > n) | (k >= points)
            ck = look(r, c, skip)
            mark(v + mw, h + mw, ~skip)
        if best is None:
            best, by, bx = ck, v, h
        else:
            better = ck < best
            best, by, bx = torch.where(better, ck, best), torch.where(better, v, by), torch.where(better, h, bx)
    y, x, cost = i + by, j + bx, best
    moving = zero == 0
    for _ in range(w * w + 2):
        best, by, bx = None, None, None
        for v, h in ((-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)):
            if v == 0 and h == 0:
                ck = cost
            else:
                r, c = y + v, x + h
                skip = (r < 0) | (c < 0) | (r > n) | (c > n) | ((r - i).abs() > mw) | ((c - j).abs() > mw)
                at = (r - i + mw + w * (c - j + mw)).clamp(0, w * w - 1)
                skip = skip | seen[rows, at]
                ck = look(r, c, skip)
                mark(r - i + mw, c - j + mw, ~skip & moving)
            if best is None:
                best, by, bx = ck, zero + v, zero + h
            else:
                better = ck < best
                best, by, bx = torch.where(better, ck, best), torch.where(better, v, by), torch.where(better, h, bx)
        moving = moving & ((by != 0) | (bx != 0))
        if not bool(moving.any()):
            break
        y, x = torch.where(moving, y + by, y), torch.where(moving, x + bx, x)
        cost = torch.where(moving, best, cost)
    return y, x


def exact(case, seed):
    """The denoised frames in 64 bits where the threshold is fixed: block
    matching, one SVD per patch, overlap-add, with plain torch.  Searched
    thresholds end where the search's tolerance leaves them and have no
    value of their own."""
    c = case
    if c["call"] in ("train", "batch", "grid", "learned") or c["lam"] <= 0 or c["median"] or not c["motion"]:
        return None
    if c["step"] != 1:
        return None  # the reference's patch table indexes the edges its own way
    n, nf, bs, mw = c["n"], c["frames"], c["patch"], c["mwin"]
    nw = learned.window_length(bs, c["traj"])
    side = n - bs + 1
    if side * side * nf * nw > 400_000 or bs * bs <= c["traj"]:
        return None
    X = _frames(n, nf, c["alpha"], c["sigma"], c["mu"], c["dtype"], seed)
    X = X.to(torch.int32).double() if c["dtype"] == "u16" else X.double()
    half = nw // 2
    dev = X.device
    grid = torch.arange(side * side, device=dev)
    gi, gj = grid % side, grid // side
    q = torch.arange(bs * bs, device=dev)
    Y = torch.empty_like(X)
    for t in range(nf):
        s0 = min(max(t - half, 0), nf - nw)
        ref = t - s0
        w = X[s0:s0 + nw] / X[s0:s0 + nw].max()
        pos = [None] * nw
        pos[ref] = (gi, gj)
        zero = torch.zeros_like(gi)
        motion = {}
        passes = [(ref + k, ref + k + 1, ref + k) for k in range(nw - 1 - ref)]
        for k in range(ref):
            src, dst = ref - k, ref - k - 1
            passes.append((src, dst, dst if ref == nw - 1 and t >= nf - half else src))
        for src, dst, slot in passes:
            y, x = _arps(w[src], w[dst], gi, gj, motion.get(slot, (zero, zero)), mw, bs)
            pos[dst] = (y, x)
            motion[slot] = (y - gi, x - gj)
        M = torch.stack([w[k][(pos[k][1][:, None] + q // bs), (pos[k][0][:, None] + q % bs)] for k in range(nw)], dim=2)
        U, s, V = torch.linalg.svd(M.cpu(), full_matrices=False)
        cut = (s[:, :1] * torch.exp(-0.5 * c["lam"] * s * s)).abs() if c["expw"] else c["lam"]
        g = (s - cut).clamp(min=0.0)
        B = ((U * g[:, None, :]) @ V)[:, :, ref].to(dev)
        at = ((gj[:, None] + q // bs) * n + gi[:, None] + q % bs).reshape(-1)
        acc = torch.zeros(n * n, dtype=torch.float64, device=dev).index_add_(0, at, B.reshape(-1))
        cover = torch.zeros(n * n, dtype=torch.float64, device=dev).index_add_(0, at, torch.ones_like(B).reshape(-1))
        Y[t] = (acc / cover).reshape(n, n) * X[s0:s0 + nw].max()
    if c["call"] == "svt":
        return dict(Y=np.ascontiguousarray(Y.cpu().numpy().transpose(2, 1, 0)))
    return dict(Y=Y)
