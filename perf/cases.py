"""The calls a user of this library makes, at the sizes they make them, for timing.

Volumes are tissue phantoms like the benchmark's (nested ellipsoids, sigma-1
smoothing, 2% noise), the moving image a monotone remap of the fixed one under
a random affine or a smooth warp, generated on the GPU from the seed.

    cost      one candidate set of the affine optimiser (cost_batch)
    pairs     the candidate sets of several registrations in one launch
              (cost_batch_pairs), as the serving loop merges them
    level     a fixed number of CDM iterations at one resolution
    cdm       a whole cdm() call with the reference's schedule
    fixed     the fixed CDM schedule with gaussian field smoothing
    cdm2d     a whole 2-D cdm() call on host images
    register  one pair from host arrays to affine, field and warped image
"""
import math

import numpy as np
import torch

import tipl_amd

_context = None


def _ctx():
    """The one device context a program keeps."""
    global _context
    if _context is None:
        _context = tipl_amd.Context(0)
    return _context


def listed():
    return [
        # the ten trial steps of an L-BFGS line search at the coarse level of a
        # small pair: the smallest call, launches and latency
        {"name": "mi256-linesearch-48", "kind": "cost", "cost": "mi", "bins": 256,
         "from": "48x48x48", "to": "48x48x48", "K": 10},
        # one finite-difference gradient (12 parameters) at the half-resolution
        # level of a 182x218x182 brain: what an affine registration spends its time on
        {"name": "mi256-gradient-91", "kind": "cost", "cost": "mi", "bins": 256,
         "from": "91x109x91", "to": "91x109x91", "K": 12},
        # the coordinate grid search of one optimiser stage at full resolution,
        # 64-bin histograms (the headline benchmark) and the reference's 256 bins
        {"name": "mi64-grid-182", "kind": "cost", "cost": "mi", "bins": 64,
         "from": "182x218x182", "to": "182x218x182", "K": 64},
        {"name": "mi256-grid-182", "kind": "cost", "cost": "mi", "bins": 256,
         "from": "182x218x182", "to": "182x218x182", "K": 64},
        # same-modality registration by correlation, the fixed image larger than
        # the moving one (the cost then samples the fixed image)
        {"name": "corr-grid-uneven", "kind": "cost", "cost": "corr", "bins": 256,
         "from": "182x218x182", "to": "160x192x160", "K": 64},
        # sixteen running registrations of uneven cubes, one candidate set each
        {"name": "pairs-mi256-16", "kind": "pairs", "bins": 256, "K": 12,
         "sides": "64 75 83 96 101 110 118 128 131 139 147 155 162 173 184 192"},
        # CDM iterations at full resolution (48 of them: one level of the
        # 3 x 48 schedule below)
        {"name": "cdm-level-182", "kind": "level", "shape": "182x218x182", "iterations": 48},
        # cdm() with its defaults: a subject at template resolution, and a small pair
        {"name": "cdm-160", "kind": "cdm", "shape": "160x192x160"},
        {"name": "cdm-64", "kind": "cdm", "shape": "64x64x64"},
        # three levels, field smoothed by a sigma-2 gaussian each iteration
        {"name": "cdm-fixed-160", "kind": "fixed", "shape": "160x192x160", "levels": 3,
         "iterations": 16},
        # a single slice
        {"name": "cdm2d-218x182", "kind": "cdm2d", "shape": "218x182"},
        # the whole pipeline for one int16 pair: preprocessing, affine, CDM
        {"name": "register-96", "kind": "register", "shape": "96x96x96", "dtype": "int16"},
    ]


def _text(shape):
    return "x".join(str(n) for n in shape)


def _dims(text):
    """A shape (z, y, x) from its text."""
    return [int(n) for n in text.split("x")]


def _sides(case):
    return [int(n) for n in case["sides"].split()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, lo, hi):
    s = _log_int(rng, lo, hi)
    return [max(lo, min(hi, int(round(s * rng.uniform(0.85, 1.15))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["cost", "cost", "cost", "pairs", "level", "cdm", "fixed", "cdm2d", "register"])
    if kind == "cost":
        cost = rng.choice(["mi", "mi", "corr"])
        a = _shape(rng, 40, 182)
        b = list(a) if rng.random() < 0.5 else [max(24, int(n * rng.uniform(0.8, 1.05))) for n in a]
        return {"kind": kind, "cost": cost, "bins": rng.choice([64, 256]) if cost == "mi" else 256,
                "from": _text(a), "to": _text(b), "K": _log_int(rng, 1, 64)}
    if kind == "pairs":
        return {"kind": kind, "bins": rng.choice([64, 256]), "K": rng.randint(6, 24),
                "sides": " ".join(str(rng.randint(64, 160)) for _ in range(rng.randint(2, 12)))}
    if kind == "level":
        return {"kind": kind, "shape": _text(_shape(rng, 33, 182)), "iterations": rng.randint(8, 40)}
    if kind == "cdm":
        return {"kind": kind, "shape": _text(_shape(rng, 40, 160))}
    if kind == "fixed":
        return {"kind": kind, "shape": _text(_shape(rng, 40, 150)), "levels": rng.randint(2, 3),
                "iterations": rng.randint(6, 16)}
    if kind == "cdm2d":
        s = _log_int(rng, 64, 400)
        return {"kind": kind, "shape": _text([s, max(40, int(s * rng.uniform(0.7, 1.3)))])}
    return {"kind": kind, "shape": _text(_shape(rng, 48, 96)), "dtype": rng.choice(["int16", "float32"])}


# -- inputs ----------------------------------------------------------------------
def _axes(shape, dtype=torch.float32):
    return [torch.arange(n, device="cuda", dtype=dtype) for n in shape]


def _blur(v, sigma):
    """Separable gaussian, replicate edges."""
    r = int(math.ceil(3 * sigma))
    k = [math.exp(-0.5 * (i / sigma) ** 2) for i in range(-r, r + 1)]
    s = sum(k)
    for axis in range(v.dim()):
        n = v.shape[axis]
        out = torch.zeros_like(v)
        for i, w in zip(range(-r, r + 1), k):
            idx = torch.arange(n, device=v.device).add_(i).clamp_(0, n - 1)
            out += v.index_select(axis, idx) * (w / s)
        v = out
    return v


def _tissue(shape, gen):
    """Nested ellipsoids at 0/300/600/900, smoothed, with 2% noise."""
    u = [a * (2.0 / (n - 1)) - 1.0 for a, n in zip(_axes(shape), shape)]
    v = torch.zeros(tuple(shape), device="cuda")
    jit = ((torch.rand((3, 3), generator=gen, device="cuda") - 0.5) * 0.08).tolist()
    for cls, (r, j) in enumerate(zip(((0.85, 0.80, 0.75), (0.62, 0.58, 0.55), (0.36, 0.30, 0.33)), jit), 1):
        e = (((u[0] - j[0]) / r[0]) ** 2)[:, None, None] + (((u[1] - j[1]) / r[1]) ** 2)[None, :, None] \
            + (((u[2] - j[2]) / r[2]) ** 2)[None, None, :]
        v[e <= 1.0] = 300.0 * cls
    return _blur(v, 1.0) + torch.randn(tuple(shape), generator=gen, device="cuda") * 18.0


def _remap(v, gen):
    """A monotone cubic intensity remap of [min, max] onto itself."""
    c = torch.rand(3, generator=gen, device="cuda").tolist()
    a, b, d = 0.2 + 0.8 * c[0], 0.8 * c[1], 0.5 * c[2]
    lo, hi = v.min(), v.max()
    t = (v - lo) / (hi - lo)
    return lo + (a * t + b * t * t + d * t * t * t) / (a + b + d) * (hi - lo)


def _sample(v, coords, outside):
    """Linear interpolation at coords (one tensor per axis); outside: 'zero' or 'edge'."""
    shape = v.shape
    inside = torch.ones_like(coords[0], dtype=torch.bool)
    lo, fr = [], []
    for c, n in zip(coords, shape):
        if outside == "zero":
            inside &= (c >= 0) & (c <= n - 1)
        c = c.clamp(0, n - 1)
        i = c.floor().clamp_(max=max(n - 2, 0))
        lo.append(i.long())
        fr.append(c - i)
    out = torch.zeros_like(coords[0])
    for corner in range(1 << len(shape)):
        w = torch.ones_like(out)
        idx = torch.zeros_like(lo[0])
        for a, n in enumerate(shape):
            up = (corner >> a) & 1
            w = w * (fr[a] if up else 1 - fr[a])
            idx = idx * n + (lo[a] + up).clamp_(max=n - 1)
        out += w * v.reshape(-1)[idx]
    return torch.where(inside, out, torch.zeros_like(out)) if outside == "zero" else out


def _matrix(p, fdim, tdim):
    """From-voxel to to-voxel transform (x, y, z order) of translation, rotation,
    scaling and shear p about the grids' centres: 9 + 3 numbers."""
    cx, sx, cy, sy, cz, sz = (f(p[i]) for i in (3, 4, 5) for f in (math.cos, math.sin))
    m = np.array([[cy * cz, cy * sz, -sy],
                  [-cx * sz + sx * cz * sy, cx * cz + sx * sz * sy, sx * cy],
                  [sx * sz + cx * cz * sy, -sx * cz + cx * sz * sy, cx * cy]])
    m = m * np.asarray(p[6:9])[:, None]
    m[0] += m[1] * p[9] + m[2] * p[10]
    m[1] += m[2] * p[11]
    t = np.array(fdim[::-1], np.float64) * -0.5 + np.asarray(p[0:3])
    return m, m @ t + np.array(tdim[::-1], np.float64) * 0.5


def _affine(rng):
    """Up to 8 voxels, 10 degrees, 5% scaling, 0.03 shear."""
    r = rng.uniform(-1, 1, 12)
    return np.concatenate([8.0 * r[0:3], np.deg2rad(10.0 * r[3:6]), 1.0 + 0.05 * r[6:9], 0.03 * r[9:12]])


def _move(v, p):
    m, s = _matrix(p, v.shape, v.shape)
    z, y, x = (a.view([-1 if i == j else 1 for j in range(3)])
               for i, a in enumerate(_axes(v.shape)))
    coords = [m[r, 0] * x + m[r, 1] * y + m[r, 2] * z + s[r] for r in (2, 1, 0)]
    return _sample(v, [c.expand(v.shape).contiguous() for c in coords], "zero")


def _rbf(shape, gen, share):
    """A sum of 30 gaussian displacements (one tensor per axis), their widths an
    eighth to a quarter and the largest displacement `share` of the smallest side."""
    ax = _axes(shape)
    nd, side = len(shape), min(shape)
    d = [torch.zeros(tuple(shape), device="cuda") for _ in range(nd)]
    r = torch.rand((30, nd + 1), generator=gen, device="cuda").tolist()
    vec = torch.randn((30, nd), generator=gen, device="cuda").tolist()
    for q, v in zip(r, vec):
        sig = side * (0.125 + 0.125 * q[nd])
        w = torch.ones((), device="cuda")
        for i, a in enumerate(ax):
            g = torch.exp(-((a - q[i] * shape[i]) ** 2) / (2 * sig * sig))
            w = w * g.view([-1 if i == j else 1 for j in range(nd)])
        for i in range(nd):
            d[i] += w * v[i]
    mag = torch.sqrt(sum(c * c for c in d)).max()
    return [c * (share * side / mag) for c in d]


def _warp(v, d):
    nd = v.dim()
    coords = [a.view([-1 if i == j else 1 for j in range(nd)]) + d[i]
              for i, a in enumerate(_axes(v.shape))]
    return _sample(v, coords, "edge")


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _cost_pair(shape_from, shape_to, K, seed):
    """Fixed and moving image (float32) and K candidate transforms."""
    gen, rng = _gen(seed), np.random.default_rng(seed)
    fixed = _tissue(shape_from, gen)
    base = fixed if list(shape_to) == list(shape_from) else _tissue(shape_to, gen)
    moving = _move(_remap(base, gen), _affine(rng))
    T = np.empty((K, 12), np.float32)
    for k in range(K):
        m, s = _matrix(_affine(rng), shape_from, shape_to)
        T[k, :9], T[k, 9:] = m.reshape(9), s
    return fixed.cpu().numpy(), moving.cpu().numpy(), T


def _cdm_pair(shape, seed):
    """A phantom and its smoothly warped copy, as the CDM gets them (bytes)."""
    gen = _gen(seed)
    fixed = _tissue(shape, gen)
    moving = _warp(fixed, _rbf(shape, gen, 0.1))
    return _bytes(fixed.cpu().numpy()), _bytes(moving.cpu().numpy())


def _bytes(v):
    """Intensities scaled to 0 .. 255 in float32 and truncated."""
    lo = v.min()
    return ((v - lo) * np.float32(np.float32(255.99) / (v.max() - lo))).astype(np.uint8)


def _slice_pair(shape, seed):
    gen = _gen(seed)
    a = _blur(torch.rand(tuple(shape), generator=gen, device="cuda"), 3.0)
    b = _warp(a, _rbf(shape, gen, 0.05))
    return _bytes(a.cpu().numpy()), _bytes(b.cpu().numpy())


def _pair_list(case, seed):
    return [_cost_pair([n] * 3, [n] * 3, case["K"], seed + 977 * i)
            for i, n in enumerate(_sides(case))]


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    st = {"case": case, "ctx": ctx}
    if kind == "cost":
        f, m, st["T"] = _cost_pair(_dims(case["from"]), _dims(case["to"]), case["K"], seed)
        st["from"], st["to"] = ctx.volume(f), ctx.volume(m)
    elif kind == "pairs":
        st["pairs"] = [(ctx.volume(f), ctx.volume(m), T) for f, m, T in _pair_list(case, seed)]
    elif kind in ("level", "cdm", "fixed"):
        a, b = _cdm_pair(_dims(case["shape"]), seed)
        st["It"], st["Is"] = ctx.volume(a), ctx.volume(b)
        if kind == "fixed":
            st["param"] = ctx.cdm_param(levels=case["levels"], level_iterations=case["iterations"],
                                        field_bandwidth=8)
    elif kind == "cdm2d":
        st["It"], st["Is"] = _slice_pair(_dims(case["shape"]), seed)
    else:
        gen, rng = _gen(seed), np.random.default_rng(seed)
        fixed = _tissue(_dims(case["shape"]), gen)
        moving = _warp(_remap(fixed, gen), _rbf(_dims(case["shape"]), gen, 0.06))
        small = _affine(rng)
        small[0:3] *= min(_dims(case["shape"])) / 182.0
        dt = np.dtype(case["dtype"])
        out = []
        for v in (fixed, _move(moving, small)):
            v = v.cpu().numpy()
            out.append((np.rint(v) if dt.kind == "i" else v).astype(dt))
        st["fixed"], st["moving"] = out
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "cost":
        return ctx.cost_batch(st["from"], st["to"], st["T"], case["cost"], case["bins"])
    if kind == "pairs":
        return ctx.cost_batch_pairs(st["pairs"], "mi", case["bins"])
    if kind == "level":
        return ctx.cdm_level_iterations(st["It"], st["Is"], case["iterations"], want_field=True)
    if kind in ("cdm", "fixed"):
        return ctx.cdm(st["It"], st["Is"], st.get("param"))[1]
    if kind == "cdm2d":
        return ctx.cdm2d(st["It"], st["Is"])[1]
    r = tipl_amd.register(ctx, st["fixed"], st["moving"], nonlinear=True, preprocess="mm_reg",
                          outputs=("warped",))
    return {"T": r["T"], "field": r["field"], "warped": r["warped"],
            "r": np.array([r["cost"], r["r_linear"], r["r_nonlinear"]])}


# -- what a pass cannot do without -------------------------------------------------
# Per voxel of one CDM iteration, 3-D: compose 30, window sums 40, regression 25,
# 12 Jacobi sweeps of 7 operations on 3 components, composition of the fields 80,
# smoothing 24; 2-D: the same with 2 components and 5-point stencils.
_ITER3, _ITER2 = 30 + 40 + 25 + 252 + 80 + 24, 15 + 25 + 25 + 120 + 30 + 14


def _vox(shape):
    return int(np.prod([int(n) for n in shape]))


def work(case):
    kind = case["kind"]
    if kind in ("cost", "pairs"):
        if kind == "cost":
            sizes = [(_dims(case["from"]), _dims(case["to"]))]
        else:
            sizes = [([n] * 3, [n] * 3) for n in _sides(case)]
        nbytes = flops = 0
        for a, b in sizes:
            nbytes += _vox(a) + _vox(b) + case["K"] * (48 + 8)
            # position 6, seven linear interpolations of 2 operations
            flops += _vox(a if case.get("cost") != "corr" or _vox(a) <= _vox(b) else b) * case["K"] * 20
        return {"bytes": nbytes, "flops": flops}
    n = _vox(_dims(case["shape"]))
    if kind == "level":
        return {"bytes": 14 * n, "flops": case["iterations"] * _ITER3 * n}
    if kind == "fixed":
        voxels = sum(n // 8 ** i for i in range(case["levels"]))
        # eight rounds of the [1 2 1] filter along three axes instead of the smoothing
        return {"bytes": 14 * n, "flops": case["iterations"] * (_ITER3 - 24 + 8 * 3 * 9) * voxels}
    if kind == "cdm2d":
        # levels down to 16 pixels a side, the finest at half size, about 60 iterations each
        return {"bytes": 10 * n, "flops": 60 * _ITER2 * n // 3}
    # the levels of cdm() below full size, about 40 iterations each
    cdm = {"bytes": 14 * n, "flops": 40 * _ITER3 * n // 7}
    if kind == "cdm":
        return cdm
    item = np.dtype(case["dtype"]).itemsize
    # an affine search of about 800 evaluations, most of them at half resolution
    return {"bytes": cdm["bytes"] + (2 * item + 1) * n, "flops": cdm["flops"] + 800 * 20 * n // 6}


def tolerance(case):
    kind = case["kind"]
    if kind in ("cost", "pairs"):
        # integer sums and counts are exact.  The correlation is rounded to
        # float before 1 - r^2; the entropy is an FP64 sum of up to 65536 log terms.
        return {"rel": 1e-6} if case.get("cost") == "corr" else {"rel": 1e-11}
    if kind in ("level", "fixed"):
        # float fields whose warped image is truncated to bytes each iteration:
        # 0.03% (smoothed once an iteration) and 0.001% (eight rounds) from the
        # same loop in 64 bits
        return {"rel": 1.5e-3 if kind == "level" else 3e-4}
    if kind in ("cdm", "cdm2d"):
        # the iteration count hangs on the sign of a cost trend
        return {"rel": 5e-3}
    return {"rel": 5e-3, "differ": 0.02}


# -- the same in 64 bits -------------------------------------------------------------
def _tri(v, pos, shape):
    """Trilinear value of v (z, y, x[, channels]) at pos = (x, y, z) where
    0 <= x < w-1 and y, z alike; (value, inside)."""
    d, h, w = shape
    x, y, z = pos
    inside = (x >= 0) & (y >= 0) & (z >= 0) & (x < w - 1) & (y < h - 1) & (z < d - 1)
    x, y, z = (torch.where(inside, c, torch.zeros_like(c)) for c in pos)
    ix, iy, iz = (c.floor().long() for c in (x, y, z))
    fx, fy, fz = x - ix, y - iy, z - iz
    i0 = (iz * h + iy) * w + ix
    flat = v.reshape((d * h * w,) + v.shape[3:])
    out = 0.0
    for c in range(8):
        wt = (fx if c & 1 else 1 - fx) * (fy if c & 2 else 1 - fy) * (fz if c & 4 else 1 - fz)
        # outside samples have i0 = 0 and may point past a thin volume
        i = (i0 + (c & 1) + (w if c & 2 else 0) + (w * h if c & 4 else 0)).clamp_(max=d * h * w - 1)
        t = flat[i].double()
        out = out + t * (wt if t.dim() == wt.dim() else wt.unsqueeze(-1))
    return out, inside


def _grid(shape):
    d, h, w = shape
    z, y, x = _axes(shape, torch.float64)
    return (x.view(1, 1, w).expand(shape).reshape(-1), y.view(1, h, 1).expand(shape).reshape(-1),
            z.view(d, 1, 1).expand(shape).reshape(-1))


def _resampled(to, shape_from, T):
    """to(T p) over the from grid, truncated to a byte, 0 outside."""
    x, y, z = _grid(shape_from)
    pos = [T[3 * r] * x + T[3 * r + 1] * y + T[3 * r + 2] * z + T[9 + r] for r in range(3)]
    v, inside = _tri(to, pos, to.shape)
    return torch.where(inside, v.floor(), torch.zeros_like(v)).long()


def _mi(frm, to, T, bins):
    f = (frm.reshape(-1).long() * bins) >> 8
    t = (_resampled(to, frm.shape, T) * bins) >> 8
    H = torch.bincount(f * bins + t, minlength=bins * bins).view(bins, bins).double()
    p = H * torch.log((H / H.sum(1, keepdim=True).clamp(min=1) / H.sum(0, keepdim=True).clamp(min=1))
                      .clamp(min=1e-300))
    return -float(torch.where(H > 0, p, torch.zeros_like(p)).sum()) / (bins * bins)


def _corr(frm, to, T):
    if frm.numel() > to.numel():
        m = np.linalg.inv(T[:9].reshape(3, 3))
        frm, to, T = to, frm, np.concatenate([m.reshape(9), -m @ T[9:]])
    x = frm.reshape(-1).double()
    y = _resampled(to, frm.shape, T).double()
    x, y = x - x.mean(), y - y.mean()
    return 1.0 - float((x * y).mean() ** 2 / ((x * x).mean() * (y * y).mean()))


def _costs(f, m, T, cost, bins):
    frm, to = (torch.from_numpy(_bytes(v)).cuda() for v in (f, m))
    T = T.astype(np.float64)
    return np.array([_corr(frm, to, t) if cost == "corr" else _mi(frm, to, t, bins) for t in T])


def _neighbours(v, n, w, wh):
    """Sum over the six flat-index neighbours of v (n, 3), dropped at the array's ends."""
    s = torch.zeros_like(v)
    for o in (1, w, wh):
        if o < n:
            s[o:] += v[:-o]
            s[:-o] += v[o:]
    return s


def _window(v):
    """Sums over the border-clipped 5 x 5 x 5 window."""
    for axis in range(3):
        n = v.shape[axis]
        out = v.clone()
        for o in (1, 2):
            if o < n:
                out.narrow(axis, o, n - o).add_(v.narrow(axis, 0, n - o))
                out.narrow(axis, 0, n - o).add_(v.narrow(axis, o, n - o))
        v = out
    return v


def _gradient(js, it):
    """The regression-weighted image gradient, (voxels, 3)."""
    j, i = js.double(), it.double()
    n = _window(torch.ones_like(j))
    sx, sy = _window(j) / n, _window(i) / n
    vx, vy = _window(j * j) / n - sx * sx, _window(i * i) / n - sy * sy
    cov = _window(j * i) / n - sx * sy
    ok = (js > 0) & (it > 0) & (vx != 0) & (vy != 0) & (cov / vx > 0)
    one = torch.ones_like(vx)
    vx, vy = torch.where(ok, vx, one), torch.where(ok, vy, one)
    a = cov / vx
    s = cov * cov / vx / vy * (j * a + (sy - a * sx) - i)
    s = torch.where(ok, s, torch.zeros_like(s))
    g = torch.zeros(j.shape + (3,), dtype=torch.float64, device=j.device)
    g[:, :, 1:-1, 0] = (j[:, :, 2:] - j[:, :, :-2]) * s[:, :, 1:-1]
    g[:, 1:-1, :, 1] = (j[:, 2:] - j[:, :-2]) * s[:, 1:-1]
    g[1:-1, :, :, 2] = (j[2:] - j[:-2]) * s[1:-1]
    return g.view(-1, 3)


def _iterate(It, Is, field, iterations, speed, smooth):
    """CDM iterations on the running field (voxels, 3)."""
    shape = It.shape
    d, h, w = shape
    n, wh, k = d * h * w, w * h, -0.5 / 3.0
    grid = torch.stack(_grid(shape), -1)
    theta = 0.0
    for _ in range(iterations):
        v, inside = _tri(Is, (grid + field).unbind(-1), shape)
        js = torch.where(inside, v.floor(), torch.zeros_like(v)).to(torch.uint8)
        js = torch.where((field == 0).all(-1), Is.reshape(-1), js)
        nd = _gradient(js.view(shape), It)
        s = nd * k
        for _ in range(12):
            s = (nd - _neighbours(s, n, w, wh)) * k
        if theta == 0.0:
            theta = float(s.norm(dim=-1).max())
            if theta == 0.0:
                break
        s *= speed / theta
        v, inside = _tri((grid + field).view(shape + (3,)), (grid + s).unbind(-1), shape)
        use = inside & (s != 0).any(-1)
        field = smooth(torch.where(use.unsqueeze(-1), v - grid, field))
    return field


def _half(v):
    """Means of 2 x 2 x 2 bytes, the last plane of an odd axis repeated."""
    v = v.long()
    for axis in range(3):
        if v.shape[axis] & 1:
            v = torch.cat([v, v.narrow(axis, v.shape[axis] - 1, 1)], axis)
        v = v.unflatten(axis, (-1, 2)).sum(axis + 1)
    return (v >> 3).to(torch.uint8)


def _binomial(f, shape, rounds):
    """[1 2 1] / 4 along each axis, replicate edges, `rounds` times."""
    f = f.view(shape + (3,))
    for _ in range(rounds):
        for axis in range(3):
            n = f.shape[axis]
            lo, hi = f.narrow(axis, 0, n - 1), f.narrow(axis, 1, n - 1)
            prev = torch.cat([f.narrow(axis, 0, 1), lo], axis)
            nxt = torch.cat([hi, f.narrow(axis, n - 1, 1)], axis)
            f = (prev + 2 * f + nxt) / 4
    return f.reshape(-1, 3)


def _fixed(It, Is, levels, iterations, speed):
    shape = It.shape
    if levels > 1:
        a, b = _half(It), _half(Is)
        low = _fixed(a, b, levels - 1, iterations, speed).view(a.shape + (3,)) * 2.0
        v, inside = _tri(low, [c * 0.5 for c in _grid(shape)], a.shape)
        field = torch.where(inside.unsqueeze(-1), v, torch.zeros_like(v))
    else:
        field = torch.zeros((It.numel(), 3), dtype=torch.float64, device=It.device)
    return _iterate(It, Is, field, iterations, speed, lambda f: _binomial(f, shape, 8))


def exact(case, seed):
    kind = case["kind"]
    if kind == "cost":
        f, m, T = _cost_pair(_dims(case["from"]), _dims(case["to"]), case["K"], seed)
        return _costs(f, m, T, case["cost"], case["bins"])
    if kind == "pairs":
        return [_costs(f, m, T, "mi", case["bins"]) for f, m, T in _pair_list(case, seed)]
    if kind not in ("level", "fixed"):
        return None  # cdm() and the optimiser stop where a cost trend changes its sign
    It, Is = (torch.from_numpy(v).cuda() for v in _cdm_pair(_dims(case["shape"]), seed))
    speed = float(np.float32(0.3))
    if kind == "fixed":
        field = _fixed(It, Is, case["levels"], case["iterations"], speed)
    else:
        d, h, w = It.shape
        s = float(np.float32(0.8))
        field = torch.zeros((It.numel(), 3), dtype=torch.float64, device="cuda")
        field = _iterate(It, Is, field, case["iterations"], speed,
                         lambda f: f * (1.0 - s) + _neighbours(f, f.shape[0], w, w * h) * (s / 6.0))
    return field.view(tuple(_dims(case["shape"])) + (3,)).cpu().numpy()
