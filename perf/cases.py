"""Workloads that the framework's performance is measured on.

Each case is one program of a user of the collision operators: a cloth simulator that calls
the stateless entry points on its own tensors, a simulator whose state is resident on the
device, or a contact query on static meshes.  `listed()` names them, `draw()` gives more of
the same ranges, `prepare()` / `run()` execute one pass, `work()` says what a pass cannot do
without and `exact()` computes a pass's results in plain 64-bit torch.

Meshes are the repository's own scenes, built on the device: a cloth of grid x grid vertices
folded over itself at x = 0.5 with a small gap, either from its flat rest state ("rest") or
with the ripple of the static proximity cloth ("rippled": a cloth in the middle of a
simulation), moving by dt * N(0, sigma) per vertex; and a sleeve closing on a static body.
"""
import math

import numpy as np
import torch

import cccollisions_amd as ccc
from cccollisions_amd import scenes

DT = 1.0 / 30.0


def listed():
    return [
        # one impulse pass on the smallest mesh a program checks its set-up with: pure latency
        dict(name="pass-450", kind="pass", grid=16, fold="rest", sigma=0.5, batch=1, dtype="float64", candidates=64),
        # static proximity list of a 7,938-triangle cloth (rest state validation, self-contact)
        dict(name="proximity-8k", kind="proximity", grid=64, fold="rippled", gap=1e-3, threshold=2e-3, dtype="float64", rows=48),
        # equal-size meshes stacked in one tensor: a small batch of simulations, ragged size
        dict(name="batch-6x5k", kind="pass", grid=51, fold="rippled", sigma=0.5, batch=6, dtype="float64", candidates=96),
        # a pass restricted to the triangles that a previous pass moved (about a tenth of them)
        dict(name="partial-20k", kind="partial", grid=100, fold="rippled", sigma=0.3, share=0.1, dtype="float64", candidates=128),
        # the same pass in single precision, for simulators that run in float
        dict(name="pass-f32-33k", kind="pass", grid=130, fold="rippled", sigma=0.3, batch=1, dtype="float32", candidates=160),
        # collision list first, impulses from it after (a caller that filters or logs contacts)
        dict(name="collect-23k", kind="collect", grid=108, fold="rippled", sigma=0.3, dtype="float64", candidates=160, rows=96),
        # static triangle-triangle intersections of a crumpled cloth, single precision
        dict(name="intersect-52k", kind="intersect", grid=163, fold="rippled", gap=0.0, noise=2e-3, dtype="float32", rows=64),
        # one served request: a resident simulation of the serving population's median size,
        # order-independent sums
        dict(name="serve-20k", kind="sim", grid=100, fold="rippled", sigma=0.5, iters=10, deterministic=True, morton=0,
             shuffle=False, candidates=128),
        # a mesh from a file whose faces are in no spatial order, on fitted 30-bit trees
        dict(name="shuffled-32k", kind="sim", grid=128, fold="rest", sigma=0.5, iters=10, deterministic=False, morton=1,
             shuffle=True, candidates=192),
        # garment on body: 24k static body triangles and a 100k-triangle sleeve closing on an arm
        dict(name="garment-122k", kind="garment", body=32, rings=224, segments=223, sigma=0.3, iters=10, candidates=512),
        # the headline: ten impulse passes on the 130,050-triangle folded cloth, from rest
        dict(name="step-130k", kind="sim", grid=256, fold="rest", sigma=0.5, iters=10, deterministic=False, morton=0,
             shuffle=False, candidates=512),
        # many meshes of different sizes (2k-200k triangles) in one call
        dict(name="packed-12", kind="packed", count=12, lo=2000, hi=200000, fold="rippled", sigma=0.3, dtype="float64", candidates=512),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["pass", "pass", "pass", "partial", "proximity", "collect", "intersect", "sim", "sim", "garment", "packed"])
    fold = rng.choice(["rest", "rippled"])
    sigma = round(rng.uniform(0.1, 0.5), 3)
    grid = int(round(_log(rng, 12, 180)))
    dtype = rng.choice(["float64", "float64", "float32"])
    # candidate capacity with room for the densest drawn scene of this size
    cand = 96 + int(6e-3 * 2 * grid * grid)
    if kind == "pass":
        batch = rng.choice([1, 1, 2, 5])
        return dict(kind=kind, grid=grid if batch == 1 else min(grid, 90), fold=fold, sigma=sigma, batch=batch, dtype=dtype,
                    candidates=cand)
    if kind == "partial":
        return dict(kind=kind, grid=grid, fold=fold, sigma=sigma, share=round(_log(rng, 0.02, 0.5), 3), dtype="float64", candidates=cand)
    if kind == "proximity":
        return dict(kind=kind, grid=min(grid, 120), fold="rippled", gap=1e-3, threshold=round(rng.uniform(1.2e-3, 2e-3), 5),
                    dtype="float64", rows=64)
    if kind == "collect":
        grid = min(grid, 120)
        return dict(kind=kind, grid=grid, fold="rippled", sigma=sigma, dtype="float64", candidates=cand, rows=128)
    if kind == "intersect":
        return dict(kind=kind, grid=grid, fold="rippled", gap=0.0, noise=round(rng.uniform(1e-3, 2e-3), 5), dtype=dtype, rows=64)
    if kind == "sim":
        shuffle = rng.random() < 0.3
        return dict(kind=kind, grid=int(round(_log(rng, 24, 180))), fold=fold, sigma=sigma, iters=rng.choice([2, 5, 10]),
                    deterministic=rng.random() < 0.5, morton=1 if shuffle else 0, shuffle=shuffle, candidates=512)
    if kind == "garment":
        return dict(kind=kind, body=rng.randint(12, 32), rings=int(round(_log(rng, 60, 224))), segments=int(round(_log(rng, 60, 223))),
                    sigma=sigma, iters=rng.choice([2, 5, 10]), candidates=512)
    return dict(kind=kind, count=rng.randint(4, 12), lo=2000, hi=int(_log(rng, 20000, 150000)), fold=fold, sigma=sigma,
                dtype="float64", candidates=512)


# ---- scenes -----------------------------------------------------------------------------------

def _dtype(case):
    return torch.float32 if case.get("dtype") == "float32" else torch.float64


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _faces(nx, ny):
    i, j = torch.meshgrid(torch.arange(nx - 1, device="cuda"), torch.arange(ny - 1, device="cuda"), indexing="ij")
    v = (i * ny + j).reshape(-1)
    return torch.stack([v, v + ny, v + ny + 1, v, v + ny + 1, v + 1], 1).reshape(-1, 3)


def _cloth(grid, fold, gap=1e-3, noise=0.0, gen=None):
    """Vertices [V, 3] and faces [F, 3] of the folded cloth."""
    s = torch.linspace(0.0, 1.0, grid, dtype=torch.float64, device="cuda")
    x, y = torch.meshgrid(s, s, indexing="ij")
    x, y = x.reshape(-1), y.reshape(-1)
    right = x > 0.5
    x = torch.where(right, 1.0 - x, x)
    z = torch.where(right, gap, 0.0).to(torch.float64)
    if fold == "rippled":
        z = z + 0.05 * torch.sin(6 * x) * torch.cos(6 * y)
    v = torch.stack([x, y, z], 1)
    if fold == "rippled":
        v = v + (noise or 1e-4) * torch.randn(v.shape, generator=gen, dtype=torch.float64, device="cuda")
    return v, _faces(grid, grid)


def _moving(case, grid, gen):
    x0, f = _cloth(grid, case["fold"], gen=gen)
    x1 = x0 + DT * case["sigma"] * torch.randn(x0.shape, generator=gen, dtype=torch.float64, device="cuda")
    return x0, x1, f


def _vertex_masses(n, gen):
    return 0.5 + 1.5 * torch.rand(n, generator=gen, dtype=torch.float64, device="cuda")


def _soups(case, grid, gen, dtype):
    x0, x1, f = _moving(case, grid, gen)
    m = _vertex_masses(x0.shape[0], gen)
    return x0[f].to(dtype), x1[f].to(dtype), m[f].to(dtype)


def _packed_grids(case, gen_cpu):
    sizes = np.exp(gen_cpu.uniform(math.log(case["lo"]), math.log(case["hi"]), case["count"]))
    sizes[0], sizes[-1] = case["lo"], case["hi"]
    return [scenes.grid_size_for_triangles(int(s)) for s in sizes]


def _garment(case, seed):
    sc = scenes.garment_on_body(case["body"], case["rings"], case["segments"], seed=seed % (1 << 31), sigma=case["sigma"])
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (sc.x0, sc.x1, sc.faces, sc.corner_masses())]


def _inputs(case, seed):
    """What the case's program computes on, from the seed alone."""
    gen, dtype = _generator(seed), _dtype(case)
    kind = case["kind"]
    if kind in ("pass", "partial", "collect"):
        parts = [_soups(case, case["grid"], gen, dtype) for _ in range(case.get("batch", 1))]
        t0, t1, m = (torch.stack([p[k] for p in parts]).contiguous() for k in range(3))
        check = None
        if kind == "partial":
            # a contiguous patch, as a contact region is
            n = t0.shape[1]
            width = max(1, int(case["share"] * n))
            first = int(torch.randint(0, n - width + 1, (1,), generator=gen, device="cuda"))
            check = torch.zeros((1, n), dtype=torch.bool, device="cuda")
            check[0, first:first + width] = True
        return t0, t1, m, check
    if kind in ("proximity", "intersect"):
        v, f = _cloth(case["grid"], case["fold"], gap=case["gap"], noise=case.get("noise", 0.0), gen=gen)
        return (v[f][None].to(dtype).contiguous(),)
    if kind == "packed":
        # the sizes are the case's own (a program's meshes do not change between passes)
        parts = [_soups(case, g, gen, dtype) for g in _packed_grids(case, np.random.default_rng(4))]
        offsets = np.cumsum([0] + [p[0].shape[0] for p in parts]).tolist()
        return tuple(torch.cat([p[k] for p in parts]).contiguous() for k in range(3)) + (offsets,)
    if kind == "garment":
        return tuple(_garment(case, seed))
    x0, x1, f = _moving(case, case["grid"], gen)
    m = _vertex_masses(x0.shape[0], gen)
    if case["shuffle"]:
        f = f[torch.randperm(f.shape[0], generator=gen, device="cuda")].contiguous()
    return x0, x1, f, m[f].contiguous()


# ---- one pass ---------------------------------------------------------------------------------

def prepare(case, seed):
    inputs = _inputs(case, seed)
    sim = None
    if case["kind"] in ("sim", "garment"):
        x0, x1, f, m = inputs
        sim = ccc.Sim(x0, x1, f, m, iters=case["iters"], max_candidates=case["candidates"],
                      deterministic=case.get("deterministic", False), morton=case.get("morton", 0))
    return case, inputs, sim


def _ordered(rows, n):
    """The rows of a contact list as keys in ascending order (the list itself is in no order):
    what a program sorts by to group the contacts of a triangle."""
    r = rows[0]
    key = (r[:, 0] * n + r[:, 1]) * 16
    if r.shape[1] > 2:
        key = key + r[:, 2]
    return torch.sort(key).values


def run(state):
    case, inputs, sim = state
    kind = case["kind"]
    if sim is not None:
        sim.set_positions(inputs[0], inputs[1])
        sim.step()
        return sim.positions()[1]
    if kind == "pass":
        t0, t1, m, _ = inputs
        bb, tree = ccc.bvh_motion(t0, t1)
        return ccc.compute_impulses(bb, tree, t0, t1, m, case["candidates"], 16)
    if kind == "partial":
        t0, t1, m, check = inputs
        bb, tree = ccc.bvh_motion(t0, t1)
        return ccc.compute_impulses_partial(bb, tree, t0, t1, m, check, case["candidates"], 16)
    if kind == "collect":
        t0, t1, m, _ = inputs
        bb, tree = ccc.bvh_motion(t0, t1)
        coll, roots = ccc.find_collisions_continuous(bb, tree, t0, t1, case["candidates"], case["rows"])
        return ccc.compute_impulses_from_collisions(coll, roots, t0, t1, m)
    if kind == "packed":
        t0, t1, m, offsets = inputs
        return ccc.compute_impulses_packed(t0, t1, m, offsets, case["candidates"])
    t = inputs[0]
    bb, tree = ccc.bvh(t)
    if kind == "proximity":
        rows = ccc.find_proximity(bb, tree, t, case["threshold"], case["rows"])
        rows = rows[0] if isinstance(rows, (list, tuple)) else rows
    else:
        rows = ccc.find_collisions(bb, tree, t, 0.0, case["rows"])
    return bb, _ordered(rows, t.shape[1])


# ---- what a pass cannot do without ------------------------------------------------------------

def _cloth_counts(case, tris):
    """Estimated sub-primitive pairs of one pass on a folded cloth: those of a triangle's own
    neighbourhood and those within reach of the motion, whose number grows with the
    triangles per area (3,000 per triangle on the 130k cloth at sigma 0.5)."""
    return tris * (60 + 3000 * (tris / 130050.0) * (case["sigma"] / 0.5) ** 2)


def work(case):
    kind = case["kind"]
    size = 4 if case.get("dtype") == "float32" else 8
    passes = case.get("iters", 1)
    if kind == "garment":
        n = 24 * (case["body"] - 1) ** 2 + 2 * (case["rings"] - 1) * case["segments"]
        items = 19.9e6 * (n / 122522.0) ** 2 * (case["sigma"] / 0.3)
    elif kind == "packed":
        grids = _packed_grids(case, np.random.default_rng(4))
        sizes = [2 * (g - 1) ** 2 for g in grids]
        n, items = sum(sizes), sum(_cloth_counts(case, s) for s in sizes)
    else:
        n = 2 * (case["grid"] - 1) ** 2
        if kind in ("proximity", "intersect"):
            # soup in, boxes and rows out; every candidate pair's test
            return {"bytes": n * (9 * size + 12 * size + case["rows"] * 8.0), "flops": n * 20 * 200.0}
        items = _cloth_counts(case, n)
        if kind == "partial":
            items *= 2 * case["share"]
    batch = case.get("batch", 1)
    # t0, t1, masses in; dv, dx and the counts out; 162 flops of coefficients per pair
    return {"bytes": passes * batch * n * (39.0 * size + 12), "flops": passes * batch * items * 162.0}


# ---- the same results in plain 64-bit torch -----------------------------------------------------

_E = ((0, 1), (0, 2), (1, 2))
# corners (0-2: of the first triangle, 3-5: of the second) of the 15 sub-primitive pairs: nine
# edge-edge, face against each vertex of the second, each vertex of the first against its face
_TYPES = ([(*_E[t // 3], 3 + _E[t % 3][0], 3 + _E[t % 3][1]) for t in range(9)] + [(0, 1, 2, 3 + k) for k in range(3)]
          + [(k, 3, 4, 5) for k in range(3)])


def _exact_pairs(t0, t1, check, mesh):
    both = torch.cat([t0, t1], 1)
    lo, hi = both.amin(1), both.amax(1)
    n = lo.shape[0]
    at = torch.arange(n, device=lo.device)
    step = max(1, 40_000_000 // n)
    for a in range(0, n, step):
        i = slice(a, min(n, a + step))
        m = at[None, :] > at[i, None]
        for k in range(3):
            m &= (lo[i, k, None] <= hi[None, :, k]) & (hi[i, k, None] >= lo[None, :, k])
        if check is not None:
            m &= check[i, None] | check[None, :]
        if mesh is not None:
            m &= mesh[i, None] == mesh[None, :]
        yield (m.nonzero() + torch.tensor([a, 0], device=lo.device)).split(1_000_000)


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _dot(a, b):
    return (a * b).sum(-1)


def _cubic(c3, c2, c1, c0):
    """Real roots [m, 3] (NaN: none) of c3 t^3 + c2 t^2 + c1 t + c0."""
    nan = torch.full_like(c3, math.nan)

    def cbrt(x):
        return torch.sign(x) * x.abs() ** (1.0 / 3.0)

    f = (3 * c1 / c3 - (c2 / c3) ** 2) / 3
    g = (2 * (c2 / c3) ** 3 - 9 * c2 * c1 / c3 ** 2 + 27 * c0 / c3) / 27
    h = g * g / 4 + f ** 3 / 27
    s = c2 / (3 * c3)
    i = torch.sqrt(torch.clamp(g * g / 4 - h, min=0))
    j, k = cbrt(i), torch.acos(torch.clamp(-g / (2 * i), -1, 1)) / 3
    trig = [2 * j * torch.cos(k) - s, -j * (torch.cos(k) + math.sqrt(3.0) * torch.sin(k)) - s,
            -j * (torch.cos(k) - math.sqrt(3.0) * torch.sin(k)) - s]
    sq = torch.sqrt(torch.clamp(h, min=0))
    one = cbrt(-g / 2 + sq) + cbrt(-g / 2 - sq) - s
    roots = torch.stack([torch.where(h <= 0, trig[0], one), torch.where(h <= 0, trig[1], nan), torch.where(h <= 0, trig[2], nan)], 1)
    d = torch.sqrt(c1 * c1 - 4 * c2 * c0)
    quad = torch.stack([(-c1 + d) / (2 * c2), (-c1 - d) / (2 * c2), nan], 1)
    roots = torch.where((c3.abs() < 1e-16)[:, None], quad, roots)
    roots = torch.where(((f == 0) & (g == 0) & (h == 0))[:, None], torch.stack([-cbrt(c0 / c3), nan, nan], 1), roots)
    return torch.where(((c3 == 0) & (c2 == 0))[:, None], nan[:, None], roots)


def _weights(p, ee, inv):
    """Closest-point parameters of two edges, or barycentric (first, last) of the face, and
    the squared area they divide by."""
    if ee:
        da, db, dc = p[:, 1] - p[:, 0], p[:, 3] - p[:, 2], p[:, 2] - p[:, 0]
        c = _cross(da, db)
        den = _dot(c, c)
        return _dot(_cross(dc, db), c) / den, _dot(_cross(dc, da), c) / den, den
    face, at = ((1, 2, 3), 0) if inv else ((0, 1, 2), 3)
    e1, e2, ep = p[:, face[0]] - p[:, face[1]], p[:, face[2]] - p[:, face[1]], p[:, at] - p[:, face[1]]
    d00, d01, d11, d20, d21 = _dot(e1, e1), _dot(e1, e2), _dot(e2, e2), _dot(ep, e1), _dot(ep, e2)
    den = d00 * d11 - d01 * d01
    return (d11 * d20 - d01 * d21) / den, (d00 * d21 - d01 * d20) / den, den


def _impulse(v, d, q, t, a, b, ee, inv):
    """Impulses and position corrections [m, 4, 3] of collisions at times t."""
    p = v + d * t[:, None, None]
    nrm = _cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]) if not inv else _cross(p[:, 2] - p[:, 1], p[:, 3] - p[:, 1])
    nrm = nrm / torch.sqrt(_dot(nrm, nrm))[:, None]
    a, b = a[:, None], b[:, None]

    def mix(u, w):
        if ee:
            return u[:, 0] + (u[:, 1] - u[:, 0]) * a, w[:, 2] + (w[:, 3] - w[:, 2]) * b
        f = (1, 2, 3) if inv else (0, 1, 2)
        return u[:, f[0]] * a + u[:, f[1]] * (1 - a - b) + u[:, f[2]] * b, w[:, 0 if inv else 3]

    p0, p1 = mix(v, v)
    d0, d1 = mix(d, d)
    m0, m1 = (x[:, 0] for x in mix(q[:, :, None], q[:, :, None]))
    nrm = torch.where((_dot(p1 - p0, nrm) < 0)[:, None], -nrm, nrm)
    nvel = _dot(d1 - d0, nrm)
    if inv:
        nrm, m0, m1 = -nrm, m1, m0
    off = torch.where(nvel.abs() < 1e-15, torch.full_like(nvel, 0.1), 2 * 2e-3 / -nvel).clamp(0, 1)
    share = torch.where((m0 + m1).abs() < 1e-15, torch.full_like(m0, 0.5), m0 / (m0 + m1))
    first = (1, 1, 0, 0) if ee else ((1, 0, 0, 0) if inv else (1, 1, 1, 0))
    mag = torch.stack([nvel * (1 - share) if s else -nvel * share for s in first], 1)
    imp = nrm[:, None, :] * mag[:, :, None]
    return imp, imp * (1 - (t - off).clamp(min=0))[:, None, None]


def _exact_pass(t0, t1, mass, check=None, mesh=None):
    """dv, dx [N, 3, 3] and cnt [N, 3] of one impulse pass, in 64 bits."""
    t0, t1, mass = t0.double(), t1.double(), mass.double()
    n = t0.shape[0]
    dv, dx = torch.zeros(3 * n, 3, dtype=torch.float64, device=t0.device), torch.zeros(3 * n, 3, dtype=torch.float64, device=t0.device)
    cnt = torch.zeros(3 * n, dtype=torch.int32, device=t0.device)
    for chunks in _exact_pairs(t0, t1, check, mesh):
        for pr in chunks:
            v = torch.cat([t0[pr[:, 0]], t0[pr[:, 1]]], 1)
            shared = (v[:, :3, None] == v[:, None, 3:]).all(-1).flatten(1).any(1)
            pr, v = pr[~shared], v[~shared]
            d = torch.cat([t1[pr[:, 0]], t1[pr[:, 1]]], 1) - v
            q = torch.cat([mass[pr[:, 0]], mass[pr[:, 1]]], 1)
            ids = torch.cat([3 * pr[:, :1] + torch.arange(3, device=pr.device), 3 * pr[:, 1:] + torch.arange(3, device=pr.device)], 1)
            lo, hi = torch.minimum(v, v + d), torch.maximum(v, v + d)
            for kind, c in enumerate(_TYPES):
                ee, inv = kind < 9, kind >= 12
                s = list(c[:2] if ee else c[:1] if inv else c[:3]), list(c[2:] if ee else c[1:] if inv else c[3:])
                hit = ((lo[:, s[0]].amin(1) <= hi[:, s[1]].amax(1)) & (hi[:, s[0]].amax(1) >= lo[:, s[1]].amin(1))).all(1).nonzero()[:, 0]
                w, e, mq, at = v[hit][:, c], d[hit][:, c], q[hit][:, c], ids[hit][:, c]
                a, b = w[:, :3] - w[:, 3:], e[:, :3] - e[:, 3:]

                def det(x, y, z):
                    return _dot(x, _cross(y, z))

                c3, c0 = det(b[:, 0], b[:, 1], b[:, 2]), det(a[:, 0], a[:, 1], a[:, 2])
                c2 = det(a[:, 0], b[:, 1], b[:, 2]) + det(b[:, 0], a[:, 1], b[:, 2]) + det(b[:, 0], b[:, 1], a[:, 2])
                c1 = det(b[:, 0], a[:, 1], a[:, 2]) + det(a[:, 0], b[:, 1], a[:, 2]) + det(a[:, 0], a[:, 1], b[:, 2])
                r = _cubic(c3, c2, c1, c0)
                k, which = ((r >= 0) & (r <= 1)).nonzero(as_tuple=True)
                t, w, e, mq, at = r[k, which], w[k], e[k], mq[k], at[k]
                x, y, den = _weights(w + e * t[:, None, None], ee, inv)
                out = (x < 0) | (x > 1) | (y < 0) | (y > 1)
                if not ee:
                    out |= (1 - x - y < 0) | (1 - x - y > 1)
                ok = ~out
                t, w, e, mq, at, x, y, den = (z[ok] for z in (t, w, e, mq, at, x, y, den))
                near = 0.5 if ee else 1.0 / 3.0
                x, y = (torch.where(den.abs() < 1e-15, torch.full_like(z, near), z) for z in (x, y))
                imp, imd = _impulse(w, e, mq, t, x, y, ee, inv)
                dv.index_add_(0, at.reshape(-1), imp.reshape(-1, 3))
                dx.index_add_(0, at.reshape(-1), imd.reshape(-1, 3))
                cnt.index_add_(0, at.reshape(-1), torch.ones_like(at.reshape(-1), dtype=torch.int32))
    return dv.view(n, 3, 3), dx.view(n, 3, 3), cnt.view(n, 3)


def exact(case, seed):
    kind = case["kind"]
    # contact decisions are made on coefficients in the inputs' precision: a single-precision
    # pass takes other collisions than 64 bits would, and has no 64-bit value
    if kind in ("pass", "partial", "collect") and case["dtype"] == "float64" and case["grid"] <= 110:
        t0, t1, m, check = _inputs(case, seed)
        each = [_exact_pass(t0[b], t1[b], m[b], None if check is None else check[b]) for b in range(t0.shape[0])]
        return [torch.stack([e[0] for e in each]), torch.stack([e[1] for e in each]), None]
    if kind in ("proximity", "intersect"):
        t = _inputs(case, seed)[0][0].double()
        return [_exact_boxes(t.amin(1), t.amax(1))[None], None]
    if kind == "sim" and case["grid"] <= 110:
        x0, x1, f, m = _inputs(case, seed)
        for _ in range(case["iters"]):
            _, dx, cnt = _exact_pass(x0[f], x1[f], m)
            d, at = dx.reshape(-1, 3), f.reshape(-1)
            ok = torch.isfinite(d).all(1)
            s = torch.zeros_like(x1).index_add_(0, at[ok], d[ok])
            c = torch.zeros_like(x1[:, 0]).index_add_(0, at[ok], cnt.reshape(-1)[ok].double())
            x1 = x1 + torch.where(c[:, None] > 0, s / c.clamp(min=1)[:, None], torch.zeros_like(s))
        return x1
    return None


def _exact_boxes(lo, hi):
    """Boxes [2n - 1, 6] of the radix tree over leaf indices: internal node i covers a range of
    leaves split at its highest differing index bit."""
    n = lo.shape[0]
    out = np.empty((2 * n - 1, 6))
    leaf = torch.cat([lo, hi], 1).cpu().numpy()
    out[n - 1:] = leaf
    # ranges from the root down, level by level (node, first leaf, last leaf)
    level, levels = np.array([[0, 0, n - 1]]), []
    while len(level):
        node, a, b = level.T
        bit = np.floor(np.log2((a ^ b).astype(np.float64))).astype(np.int64)
        split = (b >> bit << bit) - 1
        left, right = np.where(a == split, n - 1 + split, split), np.where(b == split + 1, n + split, split + 1)
        levels.append((node, left, right))
        level = np.concatenate([np.stack([left, a, split], 1)[left < n - 1], np.stack([right, split + 1, b], 1)[right < n - 1]])
    for node, left, right in reversed(levels):
        out[node, :3] = np.minimum(out[left, :3], out[right, :3])
        out[node, 3:] = np.maximum(out[left, 3:], out[right, 3:])
    return torch.from_numpy(out)
