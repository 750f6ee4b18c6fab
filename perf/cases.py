"""The calls that a program on this library makes, as cases to be timed.

A case is a dict of plain values; ``listed()`` gives the named ones and
``draw(rng)`` another one of the same ranges.  ``prepare`` makes what a
program holds before the call (unaries on the device, the model, a kept
plan), ``run`` makes one pass through the public entry points, ``work`` says
what a pass cannot do without and ``exact`` evaluates it in 64 bits with plain
torch.

Inputs follow the repository's synthetic workload: log unaries N(-3, 0.5) plus
three Gaussian bumps per part, joints of the 10-part person tree with offsets
U(-40, 40), sigmas U(4, 12) px, rotation sigmas U(0.1, 0.4).
"""
import math
import random

import numpy as np
import torch

from partapp_amd import api

CHILD = (0, 1, 2, 3, 5, 6, 7, 8, 9)  # the person tree, rooted at part 4
PARENT = (1, 4, 4, 2, 4, 7, 4, 4, 8)
ROOT, P = 4, 10
LOG_ZERO = -1e6
MOST = 32 * 300 * 300 * 24  # states of the largest sweep


def listed():
    return [
        # one joint's message on a small grid: the smallest call, all latency
        dict(name="message_24x41x57", kind="message", R=24, h=41, w=57, cov="diagonal", sparse=False),
        # one message of a joint with a learned full covariance, upward (sparse) rotation
        dict(name="message_full_24x200x200", kind="message", R=24, h=200, w=200, cov="full", sparse=True),
        # one image through the reference-shaped call, which plans and runs: a small image
        dict(name="image_24x112x128", kind="image", R=24, S=1, h=112, w=128, cov="diagonal", masks=False),
        # the same at the reference's default of 48 rotations and the common image size
        dict(name="image_48x300x300", kind="image", R=48, S=1, h=300, w=300, cov="diagonal", masks=False),
        # serving one image at a time on a kept plan, captured as a graph
        dict(name="serve_bf16mix_24x160x160", kind="sweep", method="bf16mix", R=24, S=1, n=1, h=160, w=160,
             uneven=False, cov="diagonal", masks=False, guard=False, graph=True),
        # the benchmark's batch, the drop-in arithmetic and the matrix-core method
        dict(name="batch_fp32_32x300x300x24", kind="sweep", method="fp32", R=24, S=1, n=32, h=300, w=300,
             uneven=False, cov="diagonal", masks=False, guard=False, graph=False),
        dict(name="batch_bf16mix_32x300x300x24", kind="sweep", method="bf16mix", R=24, S=1, n=32, h=300, w=300,
             uneven=False, cov="diagonal", masks=False, guard=False, graph=False),
        # images of uneven odd sizes at 48 rotations, the drop-in arithmetic
        dict(name="uneven_fp32_48", kind="sweep", method="fp32", R=48, S=1, n=6, h=333, w=251, uneven=True,
             cov="diagonal", masks=False, guard=False, graph=False),
        # uneven images at three scales with an upright torso, border strips and the MAP guard
        dict(name="uneven_bf16mix_3scales_guard", kind="sweep", method="bf16mix", R=24, S=3, n=8, h=320, w=320,
             uneven=True, cov="diagonal", masks=True, guard=True, graph=False),
        # a small batch whose joints all have full covariances
        dict(name="full_fp32_4x200x200x24", kind="sweep", method="fp32", R=24, S=1, n=4, h=200, w=200,
             uneven=False, cov="full", masks=False, guard=False, graph=False),
        # before the sweep: an image's score grids to log unaries, with the DPM and torso position terms
        dict(name="unaries_24x300x300", kind="unaries", R=24, h=300, w=300, interpolate=False),
        # after it: the local maxima of all part marginals
        dict(name="local_max_24x300x300", kind="localmax", R=24, h=300, w=300, max_n=1000),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["message", "image", "sweep", "sweep", "sweep", "unaries", "localmax"])
    R = rng.choice([24, 24, 48])
    if kind == "message":
        return dict(kind=kind, R=R, h=_size(rng, 40, 480), w=_size(rng, 40, 480),
                    cov=rng.choice(["diagonal", "diagonal", "full"]), sparse=rng.random() < 0.5)
    if kind == "image":
        return dict(kind=kind, R=R, S=rng.choice([1, 1, 3]), h=_size(rng, 96, 400), w=_size(rng, 96, 400),
                    cov="diagonal", masks=rng.random() < 0.3)
    if kind == "unaries":
        return dict(kind=kind, R=R, h=_size(rng, 100, 480), w=_size(rng, 100, 480), interpolate=rng.random() < 0.5)
    if kind == "localmax":
        return dict(kind=kind, R=R, h=_size(rng, 100, 480), w=_size(rng, 100, 480),
                    max_n=rng.choice([100, 1000, 4096]))
    method = rng.choice(["fp32", "bf16mix"])
    S = rng.choice([1, 1, 3])
    uneven = rng.random() < 0.5
    h, w = _size(rng, 96, 480), _size(rng, 96, 480)
    full = rng.random() < 0.2
    # an uneven image has up to 1.5^2 times the states of an even one; a full covariance some eight times the work
    most = MOST // (R * S * h * w) // (3 if uneven else 1) // (8 if full else 1)
    n = min(_size(rng, 1, 48), max(1, most))
    return dict(kind=kind, method=method, R=R, S=S, n=n, h=h, w=w, uneven=uneven,
                cov="full" if full else "diagonal", masks=rng.random() < 0.3,
                guard=method == "bf16mix" and not full and rng.random() < 0.3, graph=rng.random() < 0.3)


# ------------------------------------------------------------------- inputs

def _joints(seed, cov):
    """Joints of the person tree as api.Joint; cov 'full' adds a correlation of +-0.45."""
    r = random.Random(seed)
    out = []
    for k, (c, p) in enumerate(zip(CHILD, PARENT)):
        oc, op = ((r.uniform(-40, 40), r.uniform(-40, 40)) for _ in range(2))
        a, b = r.uniform(4, 12) ** 2, r.uniform(4, 12) ** 2
        x = (0.45 if (k + seed) % 2 else -0.45) * math.sqrt(a * b) if cov == "full" else 0.0
        sigma, mean = r.uniform(0.1, 0.4), r.uniform(-math.pi / 6, math.pi / 6)
        out.append(api.Joint(c, p, oc, op, (a, x, x, b), mean, sigma))
    return out


def _exp_param(case):
    S = case.get("S", 1)
    strip = 0.1 if case.get("masks") else 0.0
    lo, hi = (1.0, 1.0) if S == 1 else (0.7, 1.3)
    return api.ExpParam(-180.0, 180.0, case["R"], lo, hi, S, strip)


def _upright(case):
    return [1 if case.get("masks") and p in (2, ROOT) else 0 for p in range(P)]


def _sizes(case, seed):
    """Sizes of a batch: all alike, or each side within a factor of 1.5 (a tall, a wide, ...)."""
    n, h, w = case["n"], case["h"], case["w"]
    if not case["uneven"]:
        return [(h, w)] * n
    r = random.Random(n * 1000 + h + w)  # the batch's shape belongs to the case, not to the seed
    return [tuple(max(48, min(480, int(v * r.uniform(0.67, 1.5)))) for v in (h, w)) for _ in range(n)]


def _fill_unary(out, gen):
    """Log unaries [parts][S][R][H][W] in place."""
    out.normal_(-3.0, 0.5, generator=gen)
    n, S, R, H, W = out.shape
    r = random.Random(int(torch.randint(1 << 30, (1,), generator=gen, device=out.device)))
    yy = torch.arange(H, device=out.device, dtype=torch.float32)[:, None]
    xx = torch.arange(W, device=out.device, dtype=torch.float32)[None, :]
    for p in range(n):
        for _ in range(3):
            x, y, k = r.randrange(W), r.randrange(H), r.randrange(R)
            out[p, :, k] += 4.0 * torch.exp(-((xx - x) ** 2 + (yy - y) ** 2) / 72.0)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    if kind == "message":
        child = torch.empty((1, 1, case["R"], case["h"], case["w"]), device="cuda")
        _fill_unary(child, gen)
        return dict(case=case, child=child[0, 0], joint=_joints(seed, case["cov"])[0],
                    model=api.person_model(_exp_param(case), _joints(seed, "diagonal")))
    if kind == "image":
        un = torch.empty((P, case["S"], case["R"], case["h"], case["w"]), device="cuda")
        _fill_unary(un, gen)
        model = api.person_model(_exp_param(case), _joints(seed, case["cov"]), is_upright=_upright(case))
        return dict(case=case, unary=un, model=model)
    if kind == "sweep":
        sizes = _sizes(case, seed)
        joints = [_joints(seed * 100 + i, case["cov"]) for i in range(len(sizes))]
        model = api.person_model(_exp_param(case), joints[0], is_upright=_upright(case))
        plan = api.Plan(model, sizes, joints)
        plan.set_method(case["method"])
        if case["guard"]:
            plan.set_map_guard(api.Plan.MAP_GUARD_TAU[case["method"]])
        un = torch.empty(plan.unary_numel, device="cuda")
        for i in range(len(sizes)):
            _fill_unary(plan.instance_view(un, i), gen)
        stream = torch.cuda.Stream() if case["graph"] else None
        state = dict(case=case, plan=plan, model=model, unary=un, marg=torch.empty_like(un), stream=stream,
                     root=torch.empty(plan.root_numel, device="cuda"),
                     maps=torch.zeros(plan.map_numel * 4, dtype=torch.int32, device="cuda"))
        if stream is not None:
            stream.wait_stream(torch.cuda.current_stream())
        return state
    if kind == "unaries":
        R, H, W = case["R"], case["h"], case["w"]
        side = int(math.ceil(math.hypot(H, W)))  # the detector runs on the rotated image's bounding square
        grids = torch.empty((P * R, side, side), device="cuda").normal_(0.1, 0.4, generator=gen)
        grids[torch.rand(grids.shape, generator=gen, device="cuda") < 0.05] = 0.0  # cells it did not evaluate
        dpm = torch.rand((1, H, W), generator=gen, device="cuda")
        return dict(case=case, grids=grids, dpm=dpm, Tig=_score_transforms(R, H, W, side),
                    prior=(4.0, -7.0, 0.02 * W * W, 0.02 * H * H))
    # the marginals of the parts: the unary's noise on a smooth message
    R, H, W = case["R"], case["h"], case["w"]
    grids = torch.empty((P, 1, R, H, W), device="cuda")
    _fill_unary(grids, gen)
    for p in range(P):
        m = torch.empty((1, R, H, W), device="cuda").normal_(0.0, 30.0, generator=gen)
        for _ in range(2):
            m = torch.nn.functional.avg_pool2d(m, 17, 1, 8)
        grids[p, 0] += m[0]
    return dict(case=case, grids=[grids[p, 0] for p in range(P)])


def _score_transforms(R, H, W, side):
    """Tig [P * R][3][3]: the grid of rotation r, about its centre, onto the image."""
    T = np.zeros((R, 3, 3))
    for r in range(R):
        a = math.radians(-180.0 + 360.0 / R * (r + 0.5))
        c, s, m = math.cos(a), math.sin(a), 0.5 * (side - 1)
        T[r] = [[c, -s, 0.5 * (W - 1) - c * m + s * m], [s, c, 0.5 * (H - 1) - s * m - c * m], [0, 0, 1]]
    return np.tile(T, (P, 1, 1))


# --------------------------------------------------------------------- pass

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "message":
        j = st["joint"]
        return api.compute_rot_joint_marginal(st["model"], st["child"], j.offset_c, j.offset_p, j.C, j.rot_mean,
                                              j.rot_sigma, 1.0, is_sparse=case["sparse"])
    if kind == "image":
        root, marg, best, maps = api.compute_root_posterior_rot(st["model"], st["unary"])
        return dict(root=root, marginals=marg, best=np.array([[b.rotidx, b.y, b.x] for b in best]),
                    map=np.stack([maps["rotidx"], maps["y"], maps["x"]]), score=np.ascontiguousarray(maps["score"]))
    if kind == "sweep":
        st["plan"].execute(st["unary"], st["marg"], st["root"], st["maps"], stream=st["stream"], graph=case["graph"])
        rec = st["maps"].view(-1, 4)
        return dict(marginals=st["marg"], root=st["root"], map=rec[:, :3], score=rec[:, 3].view(torch.float32))
    if kind == "unaries":
        un = api.ingest_scores(st["grids"], st["Tig"], case["interpolate"], case["h"], case["w"])
        un = un.view(P, 1, case["R"], case["h"], case["w"])
        api.add_dpm_score(un[ROOT], st["dpm"], 0.8, api.DPM_RAW)
        api.set_torso_pos_prior(un[ROOT], st["prior"], 1.0)
        return un
    found = api.find_local_max(st["grids"], case["max_n"])
    return [dict(at=np.stack([f["d"], f["x"], f["y"]]), score=np.ascontiguousarray(f["score"])) for f in found]


def _states(case):
    n = case["R"] * case.get("S", 1) * case["h"] * case["w"]
    if case["kind"] == "sweep":
        n = sum(case["R"] * case["S"] * h * w for h, w in _sizes(case, 0))
    return n


def work(case):
    """Every input read once, every output written once; the filters' multiply-adds."""
    n, R, kind = _states(case), case["R"], case["kind"]
    taps = 49 + 49 + 2 * int(3 * 0.25 / (2 * math.pi / R) + 0.5) + 1  # mean lengths of the x, y and rotation filters
    if kind == "message":
        return dict(bytes=8 * n, flops=2 * taps * n)
    if kind in ("image", "sweep"):
        return dict(bytes=8 * P * n + 4 * n // R, flops=2 * taps * 18 * n)
    if kind == "unaries":
        side = int(math.ceil(math.hypot(case["h"], case["w"])))
        return dict(bytes=4 * P * (n + R * side * side), flops=P * n)
    return dict(bytes=4 * P * n, flops=10 * P * n)


# --------------------------------------------------------------- in 64 bits

def _taps(sigma):
    k = int(math.floor(3 * sigma + 0.5))
    return [float(np.float32(math.exp(-i * i / (2 * sigma * sigma)))) for i in range(-k, k + 1)]


def _filter(g, taps, dim):
    """Truncated filter of g along dim, zero outside."""
    k, n = len(taps) // 2, g.shape[dim]
    out = g * taps[k]
    for i in range(1, k + 1):
        if i >= n:
            break
        out.narrow(dim, i, n - i).add_(g.narrow(dim, 0, n - i), alpha=taps[k - i])
        out.narrow(dim, 0, n - i).add_(g.narrow(dim, i, n - i), alpha=taps[k + i])
    return out


def _rotated(R, r, scale, v):
    a = float(np.float32((-180.0 + 360.0 / R * (0.5 + r)) * math.pi / 180.0))
    c, s = math.cos(a) * scale, math.sin(a) * scale
    return c * v[0] - s * v[1], s * v[0] + c * v[1]


def _nearest(slice2d, dx, dy):
    """out(y, x) = in at the nearest of (y + dy, x + dx), LOG_ZERO outside."""
    H, W = slice2d.shape
    ys = torch.floor(torch.arange(H, dtype=torch.float64, device="cuda") + dy + 0.5).long()
    xs = torch.floor(torch.arange(W, dtype=torch.float64, device="cuda") + dx + 0.5).long()
    out = slice2d.index_select(0, ys.clamp(0, H - 1)).index_select(1, xs.clamp(0, W - 1))
    out[(ys < 0) | (ys >= H)] = LOG_ZERO
    out[:, (xs < 0) | (xs >= W)] = LOG_ZERO
    return out


def _bilinear(g, T, h, w, zero_eps=10 * float(np.finfo(np.float32).eps)):
    """[n][h][w]: each g[i] sampled at T (x, y, 1), 0 outside; T is [2][3] or [n][2][3]."""
    n, H, W = g.shape
    T = np.broadcast_to(np.asarray(T, dtype=np.float64), (n, 2, 3))
    y, x = torch.meshgrid(torch.arange(h, dtype=torch.float64, device="cuda"),
                          torch.arange(w, dtype=torch.float64, device="cuda"), indexing="ij")
    out = torch.zeros((n, h, w), dtype=torch.float64, device="cuda")
    for i in range(n):
        if i == 0 or not np.array_equal(T[i], T[i - 1]):
            sx = T[i, 0, 0] * x + T[i, 0, 1] * y + T[i, 0, 2]
            sy = T[i, 1, 0] * x + T[i, 1, 1] * y + T[i, 1, 2]
            ix, iy = torch.floor(sx).long(), torch.floor(sy).long()
            a, b = sx - ix, sy - iy
            inside = (ix >= 0) & (ix < W) & (iy >= 0) & (iy < H)
            point = inside & (a < zero_eps) & (b < zero_eps)
            full = inside & ~point & (ix < W - 1) & (iy < H - 1)
            at = iy.clamp(0, H - 1) * W + ix.clamp(0, W - 1)
            right = iy.clamp(0, H - 1) * W + (ix + 1).clamp(0, W - 1)
            below = (iy + 1).clamp(0, H - 1) * W + ix.clamp(0, W - 1)
            both = (iy + 1).clamp(0, H - 1) * W + (ix + 1).clamp(0, W - 1)
        s = g[i].reshape(-1)
        v = (1 - b) * (1 - a) * s[at] + (1 - b) * a * s[right] + b * (1 - a) * s[below] + b * a * s[both]
        out[i] = torch.where(full, v, torch.where(point, s[at], torch.zeros_like(v)))
    return out


def _scatter(g, T, h, w):
    """[n][h][w]: every nonzero cell of g[i] at the nearest cell of T (x, y, 1); the last of a scan with x outer stays."""
    n, H, W = g.shape
    T = np.broadcast_to(np.asarray(T, dtype=np.float64), (n, 2, 3))
    y, x = torch.meshgrid(torch.arange(H, dtype=torch.float64, device="cuda"),
                          torch.arange(W, dtype=torch.float64, device="cuda"), indexing="ij")
    order = (x * H + y).long()
    out = torch.zeros((n, h, w), dtype=torch.float64, device="cuda")
    for i in range(n):
        ix = torch.floor(T[i, 0, 0] * x + T[i, 0, 1] * y + T[i, 0, 2] + 0.5).long()
        iy = torch.floor(T[i, 1, 0] * x + T[i, 1, 1] * y + T[i, 1, 2] + 0.5).long()
        ok = (g[i] != 0) & (ix >= 0) & (ix < w) & (iy >= 0) & (iy < h)
        last = torch.full((h * w,), -1, dtype=torch.long, device="cuda")
        last.scatter_reduce_(0, (iy * w + ix)[ok], order[ok], "amax")
        hit = last >= 0
        out[i].view(-1)[hit] = g[i][last[hit] % H, last[hit] // H]
    return out


def _compose(A, B):
    return np.asarray(A) @ np.asarray(B)


def _inverse(T):
    (a, b, c), (d, e, f) = T[0], T[1]
    D = a * e - d * b
    i = [[e / D, -b / D], [-d / D, a / D]]
    return np.array([[i[0][0], i[0][1], -(i[0][0] * c + i[0][1] * f)],
                     [i[1][0], i[1][1], -(i[1][0] * c + i[1][1] * f)], [0, 0, 1]])


def _space(g, C, sparse):
    """The spatial Gaussian of covariance C (row major) on every slice of g."""
    if C[1] == 0 and C[2] == 0:
        return _filter(_filter(g, _taps(math.sqrt(C[0])), 2), _taps(math.sqrt(C[3])), 1)
    H, W = g.shape[1:]
    root = math.sqrt((C[0] - C[3]) ** 2 + 4 * C[1] ** 2)
    e1, e2 = 0.5 * (C[0] + C[3] - root), 0.5 * (C[0] + C[3] + root)
    u, v = 0.5 * (C[0] - C[3] - root) / C[1], 1.0
    u, v = u / math.hypot(u, v), v / math.hypot(u, v)
    into = np.array([[u, v, 0], [-v, u, 0], [0, 0, 1.0]])
    corners = into @ np.array([[0, W - 1, 0, W - 1], [0, 0, H - 1, H - 1], [1, 1, 1, 1.0]])
    mx, my = corners[0].min(), corners[1].min()
    tw, th = int(math.ceil(corners[0].max() - mx)), int(math.ceil(corners[1].max() - my))
    back = np.array([[1, 0, mx], [0, 1, my], [0, 0, 1.0]])
    away = np.array([[1, 0, -mx], [0, 1, -my], [0, 0, 1.0]])
    if sparse:
        t = _scatter(g, _compose(away, into)[:2], th, tw)
    else:
        t = _bilinear(g, _compose(_inverse(into), back)[:2], th, tw)
    t = _filter(_filter(t, _taps(math.sqrt(e1)), 2), _taps(math.sqrt(e2)), 1)
    out = np.array([[u, -v, 0], [v, u, 0], [0, 0, 1.0]])
    return _bilinear(t, _inverse(_compose(out, back))[:2], H, W)


def _message(b, oc, op, C, mean, sigma, scale, sparse):
    R = b.shape[0]
    step = math.radians(float(np.float32(360.0) / np.float32(R)))
    shift = math.floor(-mean / step + 0.5)
    M = b.max()
    g = torch.full_like(b, LOG_ZERO)
    for r in range(R):
        if 0 <= r + shift < R:
            dx, dy = _rotated(R, r, scale, oc)
            g[r + shift] = _nearest(b[r], -dx, -dy)
    g = torch.exp(g - M)
    if sigma > 0:
        f = _taps(sigma / step)
        if len(f) >= R:
            k = R - 2 if R % 2 else R - 1
            f = f[len(f) // 2 - k // 2:][:k]
        g = sum(torch.roll(g, len(f) // 2 - j, 0) * t for j, t in enumerate(f))
    g = _space(g, [scale * scale * c for c in C], sparse)
    g = torch.where(g == 0, torch.full_like(g, LOG_ZERO), torch.log(g)) + M
    out = torch.empty_like(g)
    for r in range(R):
        dx, dy = _rotated(R, r, scale, op)
        out[r] = _nearest(g[r], dx, dy)
    return out


def _sweep_exact(case, unary, joints):
    """(marginals [P][S][R][H][W], best score [S][P]).  The root posterior is
    left out: the drop-in's float sum of exp over- and underflows by definition."""
    S, R = case["S"], case["R"]
    ep = _exp_param(case)
    H, W = unary.shape[3:]
    marg = torch.empty(unary.shape, dtype=torch.float64, device="cuda")
    bins = [-180.0 + 360.0 / R * (0.5 + r) for r in range(R)]
    into = {p: [j for j in joints if j.parent_idx == p] for p in range(P)}
    for s in range(S):
        scale = ep.scale_from_index(s)
        u = unary[:, s].double()
        if case["masks"]:
            for p in (2, ROOT):
                u[p, [r for r in range(R) if not abs(bins[r]) < 15.0]] = LOG_ZERO
            k = int(float(np.float32(0.1)) * W)
            u[ROOT, :, :, :k] = LOG_ZERO
            u[ROOT, :, :, W - k:] = LOG_ZERO
        up = {}

        def belief(p):
            b = u[p].clone()
            for j in into[p]:
                up[j.child_idx] = _message(belief(j.child_idx), j.offset_c, j.offset_p, j.C, j.rot_mean, j.rot_sigma,
                                           scale, True)
                b += up[j.child_idx]
            marg[p, s] = b
            return b

        def down(p, source):
            for j in into[p]:
                m = _message(source(j), j.offset_p, j.offset_c, j.C, -j.rot_mean, j.rot_sigma, scale, False)
                c = j.child_idx
                marg[c, s] += m
                down(c, lambda _j, c=c, m=m: u[c] + m)

        belief(ROOT)
        down(ROOT, lambda j: u[ROOT] + sum(up[k.child_idx] for k in into[ROOT] if k is not j))
    return marg, marg.amax(dim=(2, 3, 4)).t()


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "message":
        j = st["joint"]
        return _message(st["child"].double(), j.offset_c, j.offset_p, j.C, j.rot_mean, j.rot_sigma, 1.0,
                        case["sparse"])
    if kind == "image":
        marg, score = _sweep_exact(case, st["unary"], st["model"].joints)
        return dict(root=None, marginals=marg, best=None, map=None, score=score)
    if kind == "sweep":
        plan = st["plan"]
        parts = []
        for i in range(plan.n_instances):
            joints = _joints(seed * 100 + i, case["cov"])
            parts.append(_sweep_exact(case, plan.instance_view(st["unary"], i), joints))
        marg, score = (torch.cat([q[k].reshape(-1) for q in parts]) for k in range(2))
        # the matrix-core method writes LOG_ZERO in tails some e^-26 below a message's maximum
        return dict(marginals=marg if case["method"] == "fp32" else None, root=None, map=None, score=score)
    if kind == "unaries":
        R, H, W = case["R"], case["h"], case["w"]
        g, T = st["grids"].double(), st["Tig"]
        un = _bilinear(g, np.stack([_inverse(t)[:2] for t in T]), H, W) if case["interpolate"] else \
            _scatter(g, T[:, :2], H, W)
        un = torch.where(un < 0, torch.full_like(un, 1e-4), un)
        un = torch.where(un == 0, torch.full_like(un, LOG_ZERO), torch.log(un)).view(P, 1, R, H, W)
        d = st["dpm"][0].double()
        un[ROOT] += torch.where(d > 1e-4, 0.8 * torch.log(d), torch.full_like(d, math.log(1e-4)))
        mx, my, vx, vy = st["prior"]
        x = 0.5 * W - torch.arange(W, dtype=torch.float64, device="cuda")[None, :]
        y = 0.5 * H - torch.arange(H, dtype=torch.float64, device="cuda")[:, None]
        score = torch.exp(-0.5 * (x - mx) ** 2 / vx) * torch.exp(-0.5 * (y - my) ** 2 / vy)
        un[ROOT] += torch.log(torch.clamp(score, min=1e-4))
        return un
    out = []
    for g in st["grids"]:
        D, H, W = g.shape
        keep = g >= torch.nn.functional.max_pool2d(g[None], 3, 1, 1)[0]
        keep[1:] &= g[:-1] < g[1:]
        keep[:-1] &= g[1:] < g[:-1]
        at = keep.transpose(1, 2).nonzero()  # d, then x, then y
        v = g[at[:, 0], at[:, 2], at[:, 1]]
        if len(v) > case["max_n"]:
            v = torch.sort(v, descending=True, stable=True).values[:case["max_n"]]
        out.append(dict(at=None, score=v.double()))
    return out
