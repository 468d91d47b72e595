"""Performance cases: the work users have this library do, through its public
entry points, over the range of sizes and options it serves.

listed() gives the named cases, draw() more of the same ranges.  prepare()
makes what a program holds before the call (the points, a resident cloud or
batch, output buffers), run() is one pass, work() the bytes and operations a
pass cannot do without, exact() the outputs in plain torch double precision.

Clouds are the library's seeded synthetic airborne tiles (terrain, vegetation,
buildings; LAS-quantized coordinates unless a case says otherwise).
"""
import math

import numpy as np
import torch

import gpupdal_amd as g
from gpupdal_amd.las import las_image

F_ALL = g.F_ALL10

# One context (and one serving loop) for the process, as a program keeps them.
_ctx = None
_server = None


def context():
    global _ctx
    if _ctx is None:
        _ctx = g.Context(0)
    return _ctx


def server():
    global _server
    if _server is None:
        _server = g.Server(0, workers=2)
    return _server


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # A small tile through host arrays, the whole life of a cloud: upload,
        # one stage with its default knn, columns back, release.  What an
        # interactive tool or a per-tile pipeline step does.
        dict(name="host_tile_3k_normal8", kind="host", n=3001, knn=8, stages="normal",
             density=16.0),
        # A mid-size block already in device memory, no allocation allowed (a
        # caller's own loop over chunks).
        dict(name="noalloc_48k_knn16", kind="noalloc", n=48_000, knn=16,
             stages="normal+covfeat", density=16.0),
        # All ten features of a resident cloud at covariancefeatures' default
        # knn; coordinates off the LAS lattice (registered terrestrial scans).
        dict(name="cloud_250k_all10_knn10", kind="cloud", n=250_000, knn=10, stages="all10",
             density=12.0, quantum=1e-7),
        # The benchmark's step: normal + covariancefeatures, one 4M-point
        # airborne tile.
        dict(name="cloud_4m_knn16", kind="cloud", n=4_000_000, knn=16,
             stages="normal+covfeat", density=16.0),
        # The precision-stress mix at a large size: planar roofs and wires
        # (many exact distance ties), eigenvalues + covariancefeatures knn=32.
        dict(name="cloud_10m_roofs_knn32", kind="cloud", n=10_000_000, knn=32,
             stages="eigenvalues+covfeat", density=16.0, roof=0.05, wire=0.02),
        # A strided neighborhood (covariancefeatures stride=3) of an odd-sized
        # cloud.
        dict(name="cloud_777k_knn8_stride3", kind="cloud", n=777_777, knn=8, stride=3,
             stages="covfeat", density=25.0),
        # Many uneven tiles as one batch, knn 8 / 16 / 32 by tile.
        dict(name="batch_64_tiles", kind="batch", n=8_000_000, tiles=64, knn=0,
             stages="normal+covfeat", density=0.0),
        # Radius neighborhoods (the stages' radius option).
        dict(name="radius_1m_r1", kind="radius", n=1_000_000, radius=1.0,
             stages="normal+covfeat", density=12.0),
        # Neighborhoods beyond the grid search's 63 entries.
        dict(name="cloud_150k_knn100", kind="cloud", n=150_001, knn=100,
             stages="normal+covfeat", density=16.0),
        # Per-point scale selection, results on the host.
        dict(name="optimal_1m_k10_14", kind="optimal", n=1_000_000, kmin=10, kmax=14,
             density=16.0),
        # readers.las -> filters.outlier (statistical, mean_k 8) on a file image.
        dict(name="las_outlier_2m", kind="las_outlier", n=2_000_000, knn=8, density=16.0),
        # A burst of tile requests into the serving loop, host arrays in and out.
        dict(name="serve_12_tiles", kind="serve", n=1_500_000, tiles=12, knn=10,
             stages="normal", density=16.0),
    ]


def _log_n(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed kinds with other sizes, options and densities."""
    kind = rng.choice(["host", "noalloc", "cloud", "cloud", "cloud", "batch", "radius", "large",
                       "optimal", "las_outlier", "lists", "serve"])
    density = round(math.exp(rng.uniform(math.log(2.0), math.log(50.0))), 2)
    stages = rng.choice(["normal", "covfeat", "normal+covfeat", "eigenvalues+covfeat", "all10"])
    if kind == "host":
        return dict(kind=kind, n=_log_n(rng, 1000, 30_000), knn=rng.choice([8, 10, 16]),
                    stages=stages, density=density)
    if kind == "noalloc":
        return dict(kind=kind, n=_log_n(rng, 5000, 65_536), knn=rng.choice([8, 10, 16, 24]),
                    stages=stages, density=density)
    if kind == "batch":
        return dict(kind=kind, n=_log_n(rng, 300_000, 6_000_000), tiles=rng.randint(5, 80),
                    knn=0, stages=rng.choice(["normal", "covfeat", "normal+covfeat"]),
                    density=0.0)
    if kind == "radius":
        return dict(kind=kind, n=_log_n(rng, 20_000, 2_000_000),
                    radius=round(math.sqrt(rng.uniform(8.0, 40.0) / (math.pi * density)), 3),
                    stages=stages, density=density)
    if kind == "large":
        return dict(kind="cloud", n=_log_n(rng, 10_000, 200_000), knn=rng.randint(63, 150),
                    stages=stages, density=density)
    if kind == "optimal":
        kmin = rng.randint(6, 12)
        return dict(kind=kind, n=_log_n(rng, 20_000, 1_500_000), kmin=kmin,
                    kmax=kmin + rng.randint(2, 12), density=density)
    if kind == "las_outlier":
        return dict(kind=kind, n=_log_n(rng, 50_000, 3_000_000), knn=rng.randint(4, 16),
                    density=density)
    if kind == "lists":
        return dict(kind=kind, n=_log_n(rng, 10_000, 1_000_000), knn=rng.randint(5, 40),
                    density=density)
    if kind == "serve":
        return dict(kind=kind, n=_log_n(rng, 100_000, 2_000_000), tiles=rng.randint(3, 12),
                    knn=rng.choice([8, 10, 16]), stages="normal", density=density)
    knn = rng.choice([5, 8, 10, 13, 16, 20, 24, 32, 48])
    case = dict(kind=kind, n=_log_n(rng, 20_000, 6_000_000), knn=knn, stages=stages,
                density=density)
    if stages != "normal+covfeat" and "normal" not in stages and knn <= 16 and rng.random() < 0.3:
        case["stride"] = 2
    if rng.random() < 0.3:
        case["roof"], case["wire"] = 0.05, 0.02
    if rng.random() < 0.25:
        case["quantum"] = 1e-7
    return case


# ----------------------------------------------------------------- inputs --
def _stages(case, knn=None):
    knn = case.get("knn", 8) if knn is None else knn
    stride, radius = case.get("stride", 1), case.get("radius", 0.0)
    make = {
        "normal": lambda: g.stage(g.STAGE_NORMAL, knn, radius=radius),
        "covfeat": lambda: g.stage(g.STAGE_COVFEAT, knn, stride=stride, radius=radius),
        "eigenvalues": lambda: g.stage(g.STAGE_EIGENVALUES, knn, stride=stride, radius=radius),
        "all10": lambda: g.stage(g.STAGE_COVFEAT, knn, stride=stride, radius=radius,
                                 features=F_ALL),
    }
    return [make[s]() for s in case["stages"].split("+")]


def _points(case, seed, n=None, index=0, density=None):
    n = case["n"] if n is None else n
    density = case["density"] if density is None else density
    return g.synth_cloud(n, seed=(seed * 1009 + index) * 2 + 1, side=math.sqrt(n / density),
                         roof_frac=case.get("roof", 0.0), wire_frac=case.get("wire", 0.0),
                         quantum=case.get("quantum", 0.01))


def _tiles(case):
    """Sizes, densities and knn of a batch's (or a burst's) tiles: log-uniform
    over a factor of forty, from the case alone."""
    r = np.random.default_rng(case["tiles"] * 7919 + case["n"])
    w = np.exp(r.uniform(0.0, math.log(40.0), case["tiles"]))
    sizes = np.maximum((case["n"] * w / w.sum()).astype(np.int64), 200)
    dens = r.uniform(2.0, 50.0, case["tiles"]) if not case["density"] else np.full(
        case["tiles"], case["density"])
    knn = r.choice([8, 16, 32], case["tiles"]) if not case["knn"] else np.full(
        case["tiles"], case["knn"])
    return sizes, dens, knn.astype(np.int32)


def _device_outputs(stages, n):
    cols = [torch.zeros(n, dtype=torch.float64, device="cuda")
            for _ in range(sum(g.stage_columns(s) for s in stages))]
    status = [torch.zeros(n, dtype=torch.uint8, device="cuda") for _ in stages]
    torch.cuda.synchronize()
    return cols, status


class _State:
    """What the program holds; a resident cloud or batch is let go with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    if kind == "batch":
        sizes, dens, knn = _tiles(case)
        tiles = [_points(case, seed, int(n), i, d) for i, (n, d) in enumerate(zip(sizes, dens))]
        st = _stages(case, 16)
        batch = ctx.batch(tiles)
        cols, status = _device_outputs(st, batch.n)
        return _State(case=case, batch=batch, stages=st, knn=knn, cols=cols, status=status)
    if kind == "serve":
        sizes, dens, knn = _tiles(case)
        tiles = [_points(case, seed, int(n), i, d) for i, (n, d) in enumerate(zip(sizes, dens))]
        server()
        return _State(case=case, tiles=tiles, stages=_stages(case), knn=knn)
    x, y, z = _points(case, seed)
    if kind == "host":
        return _State(case=case, xyz=(x, y, z), stages=_stages(case))
    if kind == "noalloc":
        st = _stages(case)
        dev = [torch.from_numpy(v).cuda() for v in (x, y, z)]
        cols, status = _device_outputs(st, len(x))
        return _State(case=case, dev=dev, stages=st, cols=cols, status=status)
    if kind == "las_outlier":
        lo = [float(np.floor(v.min())) for v in (x, y, z)]
        image, _ = las_image(x, y, z, offset=tuple(lo), point_format=1)
        return _State(case=case, image=image)
    cloud = ctx.cloud(x, y, z)
    if kind in ("optimal", "lists"):
        return _State(case=case, cloud=cloud)
    st = _stages(case)
    cols, status = _device_outputs(st, len(x))
    return _State(case=case, cloud=cloud, stages=st, cols=cols, status=status)


def _ptrs(tensors):
    return [t.data_ptr() for t in tensors]


# -------------------------------------------------------------------- run --
def run(s):
    """One pass.  Resident clouds and batches start from their points: the
    index is dropped first, as for points that have just arrived."""
    case, ctx = s.case, context()
    kind = case["kind"]
    if kind == "host":
        cloud = ctx.cloud(*s.xyz)
        cols, status = cloud.run(s.stages)
        cloud.close()
        return [c for per in cols for c in per] + status
    if kind == "noalloc":
        rc = ctx.run_noalloc(*_ptrs(s.dev), case["n"], s.stages, _ptrs(s.cols), _ptrs(s.status))
        if rc != g.GF_OK:
            raise RuntimeError(f"run_noalloc: {rc}")
        return s.cols + s.status
    if kind == "batch":
        s.batch.invalidate()
        s.batch.run_device(s.stages, _ptrs(s.cols), _ptrs(s.status), tile_knn=s.knn)
        return s.cols + s.status
    if kind == "serve":
        srv = server()
        tickets = [srv.submit(*t, s.stages, int(k)) for t, k in zip(s.tiles, s.knn)]
        out = []
        for t in tickets:
            cols, status, _ = srv.result(t)
            out += [c for per in cols for c in per] + status
        return out
    if kind == "las_outlier":
        cloud = ctx.cloud_from_las(s.image)
        flags, threshold = cloud.outlier("statistical", mean_k=case["knn"])
        cloud.close()
        return [flags, threshold]
    s.cloud.invalidate()
    if kind == "optimal":
        return list(s.cloud.optimal_neighborhood(case["kmin"], case["kmax"]))
    if kind == "lists":
        return list(s.cloud.knn(case["knn"]))
    s.cloud.run_device(s.stages, _ptrs(s.cols), _ptrs(s.status))
    return s.cols + s.status


# ------------------------------------------------------------- work, bounds --
def work(case):
    """Each point read once and each output written once; per point the k
    distances (8 operations), the covariance (15 per neighbor) and one 3x3
    eigensolve (about 250)."""
    n, kind = case["n"], case["kind"]
    if kind == "optimal":
        solves = case["kmax"] - case["kmin"] + 1
        return {"bytes": n * (24 + 16), "flops": n * (23.0 * case["kmax"] + 250.0 * solves)}
    if kind == "lists":
        return {"bytes": n * (24 + 4 * case["knn"] + 1), "flops": n * 8.0 * case["knn"]}
    if kind == "las_outlier":
        return {"bytes": n * (28 + 1), "flops": n * 13.0 * case["knn"]}
    st = _stages(case, 16 if kind == "batch" else None)
    out = sum(8 * g.stage_columns(s) + 1 for s in st)
    if kind in ("batch", "serve"):
        sizes, _, knn = _tiles(case)
        return {"bytes": float(sizes.sum()) * (24 + out),
                "flops": float((sizes * (23.0 * (knn + 1) + 250.0)).sum())}
    if kind == "radius":
        k = math.pi * case["radius"] ** 2 * case["density"]
    else:
        k = (case["knn"] + 1) * case.get("stride", 1)
    return {"bytes": n * (24 + out), "flops": n * (23.0 * k + 250.0)}


def tolerance(case):
    """Neighbor ids, statuses and flags are whole and do not vary.  Columns
    are double precision throughout; against exact() on points with no
    distance ties the worst is off by 5e-10 to 2e-9 (2-norm) where a small
    eigenvalue or a nearly degenerate eigenvector magnifies the last bit of
    a covariance, and Omnivariance, the cube root of a product that holds the
    smallest eigenvalue of flat neighborhoods, by 7e-6.  A single row with
    two equal smallest eigenvalues may turn its normal freely: `max`."""
    if case["kind"] == "lists":
        return "exact"
    if case["kind"] == "las_outlier":
        return {"rel": 1e-12, "max": 1e-12, "differ": 0.0}
    if case["kind"] == "optimal":
        # Two prefixes whose entropies are equal to rounding may swap.
        return {"rel": 1e-9, "max": 1e-6, "differ": 1e-6}
    if case["stages"] == "all10":
        return {"rel": 3e-5, "max": 1e-2, "differ": 0.0}
    return {"rel": 1e-8, "max": 1e-2, "differ": 0.0}


# ------------------------------------------------------------------ exact --
_EXACT_MOST = 1_100_000  # points: some seconds; beyond it a pass over windows takes too long


def _windows(x, reach, chunk):
    """Chunks [a, b) of the points sorted by x, each with the window [lo, hi)
    of points within `reach` of it along x."""
    n = len(x)
    for a in range(0, n, chunk):
        b = min(a + chunk, n)
        lo = int(torch.searchsorted(x, x[a] - reach))
        hi = int(torch.searchsorted(x, x[b - 1] + reach, right=True))
        yield a, b, lo, hi


def _d2(p, q):
    d = (p[:, None, 0] - q[None, :, 0]).square_()
    d += (p[:, None, 1] - q[None, :, 1]).square_()
    d += (p[:, None, 2] - q[None, :, 2]).square_()
    return d


def _sorted_points(x, y, z):
    p = torch.from_numpy(np.stack([x, y, z], 1)).cuda()
    order = torch.argsort(p[:, 0], stable=True)
    return p[order].contiguous(), order


def _neighbors(p, k, density):
    """The k smallest distances of every row of p (sorted by x) and their
    rows, by brute force over windows of x wide enough for the k-th."""
    n = len(p)
    k = min(k, n)
    dist = torch.empty(n, k, dtype=torch.float64, device="cuda")
    ids = torch.empty(n, k, dtype=torch.int64, device="cuda")
    xs = p[:, 0].contiguous()
    chunk = 2048
    for a in range(0, n, chunk):
        b = min(a + chunk, n)
        reach = 2.5 * math.sqrt(k / (math.pi * density))
        while True:
            lo = int(torch.searchsorted(xs, xs[a] - reach))
            hi = int(torch.searchsorted(xs, xs[b - 1] + reach, right=True))
            if hi - lo >= k:
                d, i = torch.topk(_d2(p[a:b], p[lo:hi]), k, dim=1, largest=False, sorted=True)
                if (lo == 0 and hi == n) or float(d[:, -1].max()) < reach * reach:
                    break
            reach *= 2.0
        dist[a:b], ids[a:b] = d, i + lo
    return dist, ids


def _covariances(p, ids):
    c = torch.zeros(len(p), 3, 3, dtype=torch.float64, device="cuda")
    for a in range(0, len(p), 1 << 18):
        q = p[ids[a:a + (1 << 18)]] - p[a:a + (1 << 18), None, :]
        q = q - q.mean(1, keepdim=True)
        c[a:a + (1 << 18)] = torch.matmul(q.transpose(1, 2).contiguous(), q) / (ids.shape[1] - 1)
    return c


def _radius_covariances(p, r):
    n = len(p)
    count = torch.zeros(n, dtype=torch.int64, device="cuda")
    c = torch.zeros(n, 3, 3, dtype=torch.float64, device="cuda")
    xs = p[:, 0].contiguous()
    for a, b, lo, hi in _windows(xs, r * 1.0001, 1024):
        w = (_d2(p[a:b], p[lo:hi]) < r * r).double()
        cnt = w.sum(1)
        rel = p[lo:hi] - p[a]  # near the chunk: no cancellation against the map offset
        own = p[a:b] - p[a]
        # Moments about each row's own point.
        s1 = w @ rel - cnt[:, None] * own
        mean = s1 / cnt[:, None]
        centre = own + mean
        for u in range(3):
            for v in range(u, 3):
                du = rel[None, :, u] - centre[:, None, u]
                dv = rel[None, :, v] - centre[:, None, v]
                c[a:b, u, v] = c[a:b, v, u] = (w * du * dv).sum(1) / (cnt - 1)
        count[a:b] = cnt.long()
    return c, count


def _columns(case, cov, count, order):
    """The stages' columns from covariances (rows sorted; back to the points'
    order), rows the stages skip left at zero."""
    n = len(cov)
    scale = cov.abs().amax((1, 2))
    flat = ~(scale > 1e-12)  # zero, or the 0/0 of a lone point
    safe = torch.where(flat[:, None, None], torch.eye(3, dtype=torch.float64, device="cuda"), cov)
    # LAPACK on the host: batched 3x3 solves there are accurate to the last bits.
    ev, vec = torch.linalg.eigh(safe.cpu())
    ev, vec = ev.cuda(), vec.cuda()
    radius = case.get("radius", 0.0) > 0

    def put(col, skip):
        out = torch.zeros(n, dtype=torch.float64, device="cuda")
        out[order] = torch.where(skip, torch.zeros_like(col), col)
        return out

    def normal_component(nv, axis, skip):
        # The sign of a horizontal normal is that of a rounding error in z.
        if bool((~skip & (nv[:, 2].abs() < 1e-9)).any()):
            return None
        return put(nv[:, axis], skip)

    few = count < 3
    out = []
    for stage in case["stages"].split("+"):
        if stage == "normal":
            nv = vec[:, :, 0]
            nv = nv * torch.where(nv[:, 2:] < 0, -1.0, 1.0)
            s = ev.sum(1)
            cur = torch.where(s != 0, (ev[:, 0] / s).abs(), torch.zeros_like(s))
            out += [normal_component(nv, axis, flat | few) for axis in range(3)]
            out += [put(cur, flat | few)]
        elif stage == "eigenvalues":
            out += [put(ev[:, i], flat | (few if radius else False)) for i in range(3)]
        else:
            lam = ev.flip(1).clamp(min=0.0)
            total = lam.sum(1)
            l1, l2, l3 = torch.sqrt(lam).unbind(1)
            skip = flat | (l1 == 0) | (few if radius else False)
            # |eigenvectors| weighted by the largest, middle, smallest value
            un = (vec.flip(2).abs() * torch.stack([l1, l2, l3], 1)[:, None, :]).sum(2)
            feats = [(l1 - l2) / l1, (l2 - l3) / l1, l3 / l1, un[:, 2] / un.norm(dim=1)]
            if stage == "all10":
                entropy = -(l3 * torch.log(l3) + l2 * torch.log(l2) + l1 * torch.log(l1))
                feats += [(l1 * l2 * l3) ** (1.0 / 3.0), (l1 - l3) / l1, entropy, total,
                          l3 / total, 1 - vec[:, 2, 0].abs()]
            out += [put(f, skip) for f in feats]
    return out


def _optimal(p, dist, ids, order, kmin, kmax):
    n = len(p)
    best = torch.full((n,), float("inf"), dtype=torch.float64, device="cuda")
    radius = torch.zeros(n, dtype=torch.float64, device="cuda")
    for k in range(kmin, kmax + 1):
        ev = torch.linalg.eigvalsh(_covariances(p, ids[:, :k]).cpu()).cuda().clamp(min=0.0)
        ev = ev / ev.sum(1, keepdim=True)
        e = -(ev * torch.log(ev)).sum(1)
        less = e < best
        best = torch.where(less, e, best)
        radius = torch.where(less, dist[:, k - 1].sqrt(), radius)
    out = torch.zeros_like(radius)
    out[order] = radius
    return out


def _exact_features(case, xyz, knn, density):
    p, order = _sorted_points(*xyz)
    if case.get("radius", 0.0) > 0:
        cov, count = _radius_covariances(p, case["radius"])
    else:
        stride = case.get("stride", 1)
        k = min(knn + 1, len(p))
        _, ids = _neighbors(p, k * stride, density)
        cov = _covariances(p, ids[:, ::stride])
        count = torch.full((len(p),), k, device="cuda")
    return _columns(case, cov, count, order)


def _host(cols):
    return [None if c is None else c.cpu().numpy() for c in cols]


def exact(case, seed):
    """Neighbors by brute force, covariances, eigensystems (LAPACK) and the
    stages' formulas in double precision.  Rows whose last neighbor is tied
    with the next one take either here; the library takes the one PDAL's
    tree visits first, which no formula gives."""
    kind, n = case["kind"], case["n"]
    if n > _EXACT_MOST or kind == "lists":
        return None
    if kind in ("batch", "serve"):
        sizes, dens, knn = _tiles(case)
        parts = [_exact_features(case, _points(case, seed, int(m), i, d), int(k), d)
                 for i, (m, d, k) in enumerate(zip(sizes, dens, knn))]
        nst = case["stages"].count("+") + 1
        if kind == "serve":
            return [v for part in parts for v in _host(part) + [None] * nst]
        return [None if any(v is None for v in c) else torch.cat(c)
                for c in zip(*parts)] + [None] * nst
    x, y, z = _points(case, seed)
    if kind == "las_outlier":
        p, order = _sorted_points(x, y, z)
        d = torch.zeros(n, dtype=torch.float64, device="cuda")
        d[order] = _neighbors(p, case["knn"] + 1, case["density"])[0][:, 1:].sqrt().mean(1)
        return [None, float(d.mean() + 2.0 * d.std())]
    if kind == "optimal":
        p, order = _sorted_points(x, y, z)
        dist, ids = _neighbors(p, case["kmax"], case["density"])
        return [None, _optimal(p, dist, ids, order, case["kmin"], case["kmax"]).cpu().numpy()]
    cols = _exact_features(case, (x, y, z), case.get("knn", 0), case["density"])
    cols = _host(cols) if kind == "host" else cols
    return cols + [None] * (case["stages"].count("+") + 1)
