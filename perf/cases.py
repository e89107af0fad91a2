"""Performance cases: the calls a user of this package makes, from the smallest
to the largest, on seeded synthetic satellite views.

The paths covered are those of the reference pipeline's stages: PatchMatch
solves of one view and of batches (photometric pass, geometric-consistency
pass with the filter), the serving loop, 2.5D fusion of depth maps into a DSM
(local grid and UTM grid), and 3D fusion into a point cloud that is converted
to UTM, rasterised and median-filtered.  ``exact`` restates the fusion chains
in plain torch at 64 bits; the PatchMatch search (random draws, argmin over
hypotheses) has no such value.
"""
import math
import random

import numpy as np
import torch
import torch.nn.functional as F

from vissatsatellitestereo_amd import _lib
from vissatsatellitestereo_amd.mvs import MvsContext
from vissatsatellitestereo_amd.serving import ServeLoop

DEVICE = "cuda"
ALTITUDE = 6.0e5                     # metres, perspective cameras with f ~ 1e6 px: 0.6 m pixels
FOCAL = 1.0e6
CELL = 0.5                           # heightfield and albedo grid, metres
GEO = (30.3, -81.2, 0.0, 17, 0)      # ENU origin (lat, lon, alt), UTM zone 17 N


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _solve(name, **kw):
    c = dict(name=name, kind="solve", refs=1, srcs=8, lo=1024, hi=1024, size_seed=0, radius=5, step=1,
             iters=5, geometric=False, group=1, tile=32, graph=False)
    c.update(kw)
    return c


def listed():
    return [
        # two small crops matched against each other: a quick look, where launches and copies count
        _solve("photo_pair_256", refs=2, srcs=1, lo=256, hi=256),
        # the reference's photometric flags (radius 3, 12 iterations, per-pixel draws) on a few small
        # crops of odd sizes
        _solve("photo_ref_flags", refs=4, srcs=4, lo=481, hi=641, size_seed=2, radius=3, iters=12, group=0),
        # one ordinary view at a time, every tap of the window
        _solve("photo_plain_1024"),
        # a site of ten ordinary views in one batch, every other tap, replayed from a graph
        _solve("photo_batch_1024", refs=10, step=2, graph=True),
        # the reference's consistency flags (radius 3, 1 iteration, filter) on the same kind of crops:
        # set-up, filter and outputs weigh as much as the search
        _solve("geom_ref_flags", refs=5, srcs=4, lo=481, hi=641, size_seed=3, radius=3, iters=1, group=0,
               geometric=True),
        # a batch of crops of many sizes through the consistency pass
        _solve("geom_ragged", refs=8, srcs=7, lo=512, hi=2048, size_seed=5, step=2, geometric=True, graph=True),
        # the largest views and source lists: one view of a 2.5 km site against 20 others
        _solve("photo_large_4096", srcs=20, lo=4096, hi=4096, step=2, graph=True),
        # a large crop through the consistency pass, every tap
        _solve("geom_large_2560", srcs=16, lo=2560, hi=2560, geometric=True),
        # requests of several sizes queued together and served to the end, both passes
        dict(name="serve_mixed", kind="serve", refs=6, srcs=5, lo=400, hi=1100, size_seed=7, radius=5, step=2,
             iters=5, geometric=True, group=1, tile=32, graph=False),
        # the DSM of an ordinary site from its filtered depth maps, with the per-view DSMs, as the
        # aggregation stage asks for them
        dict(name="fuse_dsm_10", kind="dsm", refs=10, lo=1024, hi=1024, size_seed=0, res=0.5, utm=False,
             per_view=True),
        # the DSM of the largest site on the UTM grid
        dict(name="fuse_dsm_40_utm", kind="dsm", refs=40, lo=4096, hi=4096, size_seed=0, res=0.3, utm=True,
             per_view=False),
        # the point cloud of a site and the DSM made from it
        dict(name="points_dsm_8", kind="points", refs=8, lo=900, hi=1024, size_seed=9, res=0.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("photo", "geom", "serve", "dsm", "points"), (40, 25, 8, 14, 13))[0]
    seed = rng.randrange(1 << 16)
    if kind in ("photo", "geom", "serve"):
        side = _log_int(rng, 160, 3072)
        c = dict(kind="serve" if kind == "serve" else "solve", refs=_log_int(rng, 1, 10),
                 srcs=_log_int(rng, 1, 20), lo=side, hi=side + rng.randrange(0, side), size_seed=seed,
                 radius=rng.choice((3, 4, 5, 5, 7)), step=rng.choice((1, 2)), iters=_log_int(rng, 1, 12),
                 geometric=kind == "geom" or (kind == "serve" and rng.random() < 0.5),
                 group=rng.choice((0, 1, 1)), tile=rng.choice((16, 32, 32, 64)),
                 graph=kind != "serve" and rng.random() < 0.5)
        if c["kind"] == "serve":
            c["refs"] = max(2, c["refs"])
            c["srcs"] = min(c["srcs"], c["refs"] - 1) if c["geometric"] else c["srcs"]
        if c["srcs"] > 16 and c["tile"] == 64:
            c["tile"] = 32
        while c["lo"] > 160 and (work(c)["flops"] > 4e12 or _images(c) * c["hi"] ** 2 > 1.2e8):
            c["lo"], c["hi"] = max(160, int(c["lo"] * 0.8)), max(161, int(c["hi"] * 0.8))
        while work(c)["flops"] > 4e12 and (c["refs"] > 2 or c["iters"] > 1):
            c["refs"], c["iters"] = max(2, c["refs"] - 1), max(1, c["iters"] - 1)
            if c["kind"] == "serve" and c["geometric"]:
                c["srcs"] = min(c["srcs"], c["refs"] - 1)
        return c
    side = _log_int(rng, 160, 3072)
    c = dict(kind=kind, refs=_log_int(rng, 3, 40) if kind == "dsm" else _log_int(rng, 4, 16), lo=side,
             hi=side + rng.randrange(0, side // 3), size_seed=seed, res=rng.choice((0.3, 0.5, 0.5, 0.8)))
    if kind == "dsm":
        c.update(utm=rng.random() < 0.5, per_view=rng.random() < 0.5)
    cap = 1.5e8 if kind == "dsm" else 1.5e7
    while c["refs"] * c["hi"] ** 2 > cap:
        c["lo"], c["hi"] = int(c["lo"] * 0.8), int(c["hi"] * 0.8)
    return c


def _images(case):
    if case["kind"] in ("dsm", "points"):
        return case["refs"]
    if case["kind"] == "serve" and case["geometric"]:
        return case["refs"]          # every source is a request of its own
    return max(case["refs"], case["srcs"] + 1)


def _sizes(case):
    """(width, height) per image: sides between lo and hi."""
    r = random.Random(case["size_seed"])
    return [(r.randint(case["lo"], case["hi"]), r.randint(case["lo"], case["hi"])) for _ in range(_images(case))]


def _sources(case, i):
    n = _images(case)
    return [(i + 1 + k) % n for k in range(case["srcs"])]


def work(case):
    sizes = _sizes(case)
    px = [w * h for w, h in sizes]
    if case["kind"] in ("solve", "serve"):
        taps = (2 * case["radius"] // case["step"] + 1) ** 2
        s = case["srcs"]
        # current plane against every source, seven candidates against the distinct sources of 15 draws
        evals = s + 7 * s * (1.0 - (1.0 - 1.0 / s) ** 15)
        passes = 2 if case["kind"] == "serve" and case["geometric"] else 1
        n = sum(px[: case["refs"]])
        flops = 30.0 * taps * evals * case["iters"] * n * passes
        # images once, 16 bytes of hypothesis, 4 of cost and 4 per source read and written per
        # iteration, depth and normal out (and the mask of the filter)
        state = 2.0 * (20 + 4 * s) * case["iters"] * n * passes
        return {"bytes": sum(px) + state + 20.0 * n, "flops": flops}
    cells = _grid(case)[4] * _grid(case)[5]
    if case["kind"] == "dsm":
        # depth in, the stack of per-view rasters (returned when asked for) and the fused cell out
        return {"bytes": 4.0 * sum(px) + (4.0 * case["refs"] + 4.0) * cells,
                "flops": (700.0 if case["utm"] else 40.0) * sum(px) + 60.0 * case["refs"] * cells}
    # depth, normal and grey in; a third of the pixels come out as points (37 bytes), which are read
    # again and written in UTM (24 + 24), rasterised (24) and filtered (8 + 4 per cell)
    return {"bytes": 17.0 * sum(px) + 0.3 * sum(px) * 109 + 16.0 * cells,
            "flops": 120.0 * case["refs"] * sum(px) + 250.0 * sum(px)}


# ---------------------------------------------------------------------------
# synthetic scene: terrain and box buildings, seen by cameras 600 km away
# ---------------------------------------------------------------------------
def _noise_field(gen, n, waves):
    out = torch.zeros((1, 1, n, n), device=DEVICE)
    for wave, amp in waves:
        m = max(2, int(n * CELL / wave) + 2)
        g = torch.randn((1, 1, m, m), generator=gen, device=DEVICE)
        out += amp * F.interpolate(g, size=(n, n), mode="bicubic", align_corners=True)
    return out


class _Scene:
    def __init__(self, sizes, seed):
        side = max(max(s) for s in sizes)
        self.half = 0.5 * 0.64 * side + 60.0
        n = int(2 * self.half / CELL) + 1
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        H = _noise_field(gen, n, ((180.0, 6.0), (60.0, 2.0), (25.0, 0.5)))
        rng = np.random.default_rng(seed)
        for _ in range(max(2, int((2 * self.half) ** 2 / 12000.0))):
            w, l = rng.uniform(10, 40, 2) / CELL
            r, c = rng.uniform(0, n, 2)
            r0, r1, c0, c1 = (max(0, int(v)) for v in (r - l / 2, r + l / 2, c - w / 2, c + w / 2))
            if r1 > r0 and c1 > c0:
                block = H[0, 0, r0:r1, c0:c1]
                block.fill_(block.mean().clamp(-25, 25) + float(rng.uniform(5, 40)))
        self.H = H
        A = _noise_field(gen, n, ((20.0, 0.5), (8.0, 0.5), (3.0, 0.6), (1.3, 0.5)))
        gy, gx = torch.gradient(H[0, 0], spacing=CELL)
        lam = ((0.25 * gy - 0.35 * gx + 0.9) / torch.sqrt(gx * gx + gy * gy + 1.0)).clamp(0.05, 1.0)
        self.A = ((0.5 + 0.17 * A[0, 0]).clamp(0.02, 1.0) * (0.35 + 0.65 * lam))[None, None]
        self.z_lo, self.z_hi = float(H.min()) - 1.0, float(H.max()) + 1.0
        self.z0 = self.z_lo - 20.0
        self.gen = gen
        self.P4, self.R = [], []
        for i, (w, h) in enumerate(sizes):
            th = math.radians(5.0 + 25.0 * ((0.61803 * i + rng.uniform(0, 0.2)) % 1.0))
            ph = math.radians(45.0 * (i % 8) + rng.uniform(-8, 8))
            d = np.array([math.sin(th) * math.sin(ph), math.sin(th) * math.cos(ph), math.cos(th)])
            C = ALTITUDE / math.cos(th) * d
            x = np.array([1.0, 0.0, 0.0]) + d * (-d[0])
            x /= np.linalg.norm(x)
            R = np.stack([x, np.cross(-d, x), -d])
            f = FOCAL / math.cos(th) * (1.0 + rng.uniform(-0.01, 0.01, 2))
            K = np.array([[f[0], rng.uniform(-20, 20), (w - 1) / 2.0 + rng.uniform(-4, 4)],
                          [0.0, f[1], (h - 1) / 2.0 + rng.uniform(-4, 4)], [0.0, 0.0, 1.0]])
            Z = ALTITUDE / math.cos(th)
            last = Z * np.array([0.0, 0.0, 1.0, -self.z0])
            self.P4.append(np.vstack([K @ np.hstack([R, (-R @ C)[:, None]]), last]))
            self.R.append(R)

    def sample(self, G, x, y):
        g = torch.stack([x / self.half, -y / self.half], -1)
        return F.grid_sample(G, g[None], mode="bilinear", padding_mode="border", align_corners=True)[0, 0]

    def depth_range(self):
        """The stretched range of the reparametrised depth, height above the reference plane."""
        return self.z_lo - self.z0 - 10.0, self.z_hi - self.z0 + 100.0

    def hit(self, i, w, h):
        """(x, y, z, depth) where each pixel's ray meets the surface."""
        Pi = np.linalg.inv(self.P4[i])
        v, u = torch.meshgrid(torch.arange(h, device=DEVICE, dtype=torch.float64),
                              torch.arange(w, device=DEVICE, dtype=torch.float64), indexing="ij")

        def at(d):
            X = [Pi[k, 0] * u + Pi[k, 1] * v + Pi[k, 2] + Pi[k, 3] * d for k in range(4)]
            return X[0] / X[3], X[1] / X[3], X[2] / X[3]

        xa, ya, za = at(0.0)
        xb, yb, zb = at(100.0)
        sx, sy = ((xb - xa) / (zb - za)).float(), ((yb - ya) / (zb - za)).float()
        x0, y0 = (xa - za * (xb - xa) / (zb - za)).float(), (ya - za * (yb - ya) / (zb - za)).float()
        del xb, yb, zb, xa, ya, za
        z = torch.full_like(x0, self.z_hi)
        for _ in range(int((self.z_hi - self.z_lo) / 1.5) + 2):     # down each ray until it is inside
            z -= 1.5 * (z > self.sample(self.H, x0 + z * sx, y0 + z * sy))
        lo, hi = z, z + 1.5
        for _ in range(6):
            mid = 0.5 * (lo + hi)
            below = mid <= self.sample(self.H, x0 + mid * sx, y0 + mid * sy)
            lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
        z = 0.5 * (lo + hi)
        x, y = x0 + z * sx, y0 + z * sy
        p2, p3 = self.P4[i][2], self.P4[i][3]
        zc = p2[0] * x.double() + p2[1] * y.double() + p2[2] * z.double() + p2[3]
        return x, y, z, ((p3[2] * z.double() + p3[3]) / zc).float()

    def image(self, x, y, z):
        a = self.sample(self.A, x + 0.37 * z, y + 0.61 * z)
        n = torch.randn(a.shape, generator=self.gen, device=DEVICE)
        return (255.0 * a + 2.0 * n).round().clamp(0, 255).to(torch.uint8)

    def estimated(self, depth, outliers, holes):
        """A depth map as a solve leaves it: noise, outliers over the range, filtered pixels 0."""
        lo, hi = self.depth_range()
        d = depth + 0.1 * torch.randn(depth.shape, generator=self.gen, device=DEVICE)
        r = torch.rand(depth.shape, generator=self.gen, device=DEVICE)
        u = torch.rand(depth.shape, generator=self.gen, device=DEVICE)
        d = torch.where(r < outliers, lo + (hi - lo) * u, d)
        return torch.where(r > 1.0 - holes, torch.zeros_like(d), d)

    def normals(self, i, shape):
        """Unit normals in camera i's frame, facing it: up with a tilt of a few degrees."""
        t = 0.05 * torch.randn(shape + (3,), generator=self.gen, device=DEVICE)
        t[..., 2] = 1.0
        n = t @ torch.tensor(self.R[i].T, dtype=torch.float32, device=DEVICE)
        return n / n.norm(dim=-1, keepdim=True)


def _grid(case):
    """(ul_e, ul_n, e_res, n_res, e_size, n_size) of the DSM around the ENU origin; the UTM grid's
    upper left corner is that of the same square about the origin's UTM coordinates."""
    half = 0.25 * 0.6 * (case["lo"] + case["hi"])
    n = int(2 * half / case["res"]) + 1
    e0 = n0 = 0.0
    if case.get("utm", case["kind"] == "points"):
        e0, n0, _ = _utm(*(torch.zeros(1, dtype=torch.float64) for _ in range(3)))
        e0, n0 = float(e0), float(n0)
    return (e0 - half, n0 + half, case["res"], case["res"], n, n)


# ---------------------------------------------------------------------------
# what a program has before the call, and the call
# ---------------------------------------------------------------------------
def prepare(case, seed):
    sizes = _sizes(case)
    sc = _Scene(sizes, seed)
    n = len(sizes)
    if case["kind"] in ("dsm", "points"):
        ctx = MvsContext(device=0)
        st = dict(case=case, ctx=ctx, ids=list(range(1, n + 1)), inv=np.linalg.inv(np.stack(sc.P4)),
                  rot=np.stack([R.T for R in sc.R]), P4=sc.P4, grid=_grid(case))
        keep = []
        for i, (w, h) in enumerate(sizes):
            x, y, z, d = sc.hit(i, w, h)
            if case["kind"] == "points":
                img = sc.image(x, y, z).cpu().numpy()
                ctx.add_image(i + 1, img, sc.P4[i])
                nrm = sc.normals(i, (h, w)).cpu().numpy()
                ctx.set_normal_map(i + 1, nrm, kind=1)
            else:
                img = nrm = None
                ctx.register_geometry(i + 1, w, h, sc.P4[i])
            d = sc.estimated(d, 0.02, 0.1).cpu().numpy()
            ctx.set_depth_map(i + 1, d, kind=1)
            if case.get("keep"):
                keep.append((d, nrm, img))
        if case["kind"] == "points" or case["utm"]:
            st["geo"] = ctx.set_geo_frame(_lib.geo_frame(*GEO))
        st["keep"] = keep
        return st
    p = dict(window_radius=case["radius"], window_step=case["step"], num_iterations=case["iters"],
             draw_group=case["group"], tile_width=case["tile"], seed=seed + 1)
    solve_geometric = case["geometric"] and case["kind"] == "solve"
    if case["geometric"]:
        p.update(geom_consistency=1, filter=1)
    ctx = MvsContext(device=0, **p)
    for i, (w, h) in enumerate(sizes):
        x, y, z, d = sc.hit(i, w, h)
        ctx.add_image(i + 1, sc.image(x, y, z).cpu().numpy(), sc.P4[i])
        if solve_geometric:          # the photometric maps, as read back from a workspace
            ctx.set_depth_map(i + 1, sc.estimated(d, 0.05, 0.0).cpu().numpy(), kind=0)
            if i < case["refs"]:
                ctx.set_normal_map(i + 1, sc.normals(i, (h, w)).cpu().numpy(), kind=0)
    views = [dict(ref=i + 1, srcs=[s + 1 for s in _sources(case, i)], depth_range=sc.depth_range())
             for i in range(case["refs"])]
    return dict(case=case, ctx=ctx, views=views)


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "solve":
        want = ("depth", "normal", "consistency") if case["geometric"] else ("depth", "normal")
        return ctx.solve(state["views"], pass_=1 if case["geometric"] else 0, want=want,
                         use_graph=case["graph"])
    if case["kind"] == "serve":
        loop = ServeLoop(ctx, want=("depth", "normal"), geometric=case["geometric"])
        tickets = [loop.submit(v) for v in state["views"]]
        loop.drain()
        return [loop.result(t) for t in tickets]
    if case["kind"] == "dsm":
        return ctx.fuse_dsm(state["grid"], state["ids"], depth_kind=1, min_measurements=3,
                            inv_proj_mats=state["inv"], per_view=case["per_view"])
    # the number of points differs from scene to scene: what stands for them is the raster of them all
    xyz, normal, grey = ctx.fuse_points(state["ids"], state["rot"], depth_kind=1, inv_proj_mats=state["inv"])
    utm = ctx.enu_to_utm(xyz)
    dsm = ctx.proj_to_grid(utm[~np.isnan(utm[:, 0])], state["grid"])
    return dict(points=len(xyz), dsm=dsm, smooth=ctx.median_blur3(dsm.astype(np.float32)))


# ---------------------------------------------------------------------------
# the fusion chains at 64 bits
# ---------------------------------------------------------------------------
def _utm(e, n, u):
    """ENU metres -> (easting, northing, altitude): WGS84, Bowring's iteration, Krueger's series to n^6."""
    lat0, lon0, alt0, zone, south = GEO
    a, f = 6378137.0, 1.0 / 298.257223563
    b, e2 = a * (1 - f), f * (2 - f)
    la, lo = math.radians(lat0), math.radians(lon0)
    N0 = a / math.sqrt(1 - e2 * math.sin(la) ** 2)
    o = ((N0 + alt0) * math.cos(la) * math.cos(lo), (N0 + alt0) * math.cos(la) * math.sin(lo),
         (N0 * (1 - e2) + alt0) * math.sin(la))
    x = o[0] - math.sin(lo) * e - math.sin(la) * math.cos(lo) * n + math.cos(la) * math.cos(lo) * u
    y = o[1] + math.cos(lo) * e - math.sin(la) * math.sin(lo) * n + math.cos(la) * math.sin(lo) * u
    z = o[2] + math.cos(la) * n + math.sin(la) * u
    p = torch.hypot(x, y)
    beta = torch.atan2(z, (1 - f) * p)
    for _ in range(5):
        phi = torch.atan2(z + e2 / (1 - e2) * b * torch.sin(beta) ** 3, p - e2 * a * torch.cos(beta) ** 3)
        beta = torch.atan2((1 - f) * torch.sin(phi), torch.cos(phi))
    alt = p * torch.cos(phi) + z * torch.sin(phi) - a * torch.sqrt(1 - e2 * torch.sin(phi) ** 2)
    lam = torch.atan2(y, x) - math.radians(6 * zone - 183)
    k = f / (2 - f)
    A = a / (1 + k) * (1 + k**2 / 4 + k**4 / 64 + k**6 / 256)
    al = (k / 2 - 2 * k**2 / 3 + 5 * k**3 / 16 + 41 * k**4 / 180 - 127 * k**5 / 288 + 7891 * k**6 / 37800,
          13 * k**2 / 48 - 3 * k**3 / 5 + 557 * k**4 / 1440 + 281 * k**5 / 630 - 1983433 * k**6 / 1935360,
          61 * k**3 / 240 - 103 * k**4 / 140 + 15061 * k**5 / 26880 + 167603 * k**6 / 181440,
          49561 * k**4 / 161280 - 179 * k**5 / 168 + 6601661 * k**6 / 7257600,
          34729 * k**5 / 80640 - 3418889 * k**6 / 1995840, 212378941 * k**6 / 319334400)
    q = math.sqrt(e2)
    t = torch.tan(phi)
    s = torch.sinh(q * torch.atanh(q * torch.sin(phi)))
    t = t * torch.sqrt(1 + s * s) - s * torch.sqrt(1 + t * t)
    xi = torch.atan2(t, torch.cos(lam))
    eta = torch.asinh(torch.sin(lam) / torch.sqrt(t * t + torch.cos(lam) ** 2))
    E, N = eta.clone(), xi.clone()
    for j, c in enumerate(al, 1):
        E += c * torch.cos(2 * j * xi) * torch.sinh(2 * j * eta)
        N += c * torch.sin(2 * j * xi) * torch.cosh(2 * j * eta)
    return 5e5 + 0.9996 * A * E, 0.9996 * A * N + (1e7 if south else 0.0), alt


def _back(Mi, u, v, d):
    X = [Mi[k, 0] * u + Mi[k, 1] * v + Mi[k, 2] + Mi[k, 3] * d for k in range(4)]
    return X[0] / X[3], X[1] / X[3], X[2] / X[3]


def _windows(a, fill):
    """The nine 3 x 3 neighbours of every cell; fill None repeats the border."""
    h, w = a.shape
    p = F.pad(a[None, None], (1, 1, 1, 1), mode="replicate")[0, 0] if fill is None else \
        F.pad(a, (1, 1, 1, 1), value=fill)
    return [p[r:r + h, c:c + w] for r in range(3) for c in range(3)]


def _median(vals):
    """Median over dim 0 of the values that are not NaN (even count: the mean of the middle two)."""
    s = torch.stack(vals) if isinstance(vals, list) else vals
    k = (~torch.isnan(s)).sum(0)
    s = torch.sort(torch.where(torch.isnan(s), torch.full_like(s, math.inf), s), 0).values
    at = lambda i: torch.gather(s, 0, i.clamp(min=0)[None])[0]  # noqa: E731
    m = 0.5 * (at((k - 1).div(2, rounding_mode="floor")) + at(k // 2))
    return torch.where(k > 0, m, torch.full_like(m, math.nan))


def _rows(fn, a, rows=512):
    """fn over bands of rows of `a` (..., rows, cols) with one row of halo on either side."""
    n, out = a.shape[-2], []
    for r in range(0, n, rows):
        lo, hi = max(0, r - 1), min(n, r + rows + 1)
        out.append(fn(a[..., lo:hi, :])[r - lo:r - lo + min(rows, n - r)])
    return torch.cat(out)


def _raster(E, N, z, g):
    r, c = torch.floor((g[1] - N) / g[2]), torch.floor((E - g[0]) / g[3])
    ok = (r >= 0) & (c >= 0) & (r < g[5]) & (c < g[4]) & torch.isfinite(z)
    cell = (r[ok] * g[4] + c[ok]).long()
    top = torch.full((g[5] * g[4],), -math.inf, dtype=torch.float64, device=z.device)
    top.scatter_reduce_(0, cell, z[ok], "amax")
    top = torch.where(torch.isinf(top), torch.full_like(top, math.nan), top).view(g[5], g[4])
    return _rows(lambda a: torch.where(torch.isnan(a), _median(_windows(a, math.nan)), a), top)


def _blur(a):
    return _rows(lambda b: _median(_windows(b, None)), a)


def _kept(case, seed):
    s = prepare(dict(case, keep=True), seed)
    s["ctx"].close()
    return s


def exact(case, seed):
    if case["kind"] == "dsm":
        return _exact_dsm(case, seed)
    if case["kind"] == "points":
        return _exact_points(case, seed)
    return None


def _exact_dsm(case, seed):
    s = _kept(case, seed)
    g = s["grid"]
    stack = []
    for Mi, (d, _, _) in zip(s["inv"], s["keep"]):
        d = torch.from_numpy(d).to(DEVICE)
        v, u = torch.nonzero(d > 0, as_tuple=True)
        E, N, z = _back(Mi, u.double(), v.double(), d[v, u].double())
        if case["utm"]:
            E, N, z = _utm(E, N, z)
        stack.append(_blur(_raster(E, N, z, g)))

    def fuse(a):
        med = _median(a)
        dev = (a - med).abs()
        # the rule drops what is further than the median deviation, itself one of the values:
        # a rounding margin keeps the values that define it
        ok = dev <= _median(dev) * (1 + 1e-9) + 1e-9
        m = torch.where(ok, a, torch.zeros_like(a)).sum(0) / ok.sum(0)
        return torch.where((~torch.isnan(a)).sum(0) >= 3, m, torch.full_like(m, math.nan))

    # per-view DSMs are 32-bit rasters by definition of the chain
    rows = max(1, int(2e8 / (len(stack) * g[4])))
    out = _blur(torch.cat([fuse(torch.stack([a[r:r + rows].float().double() for a in stack]))
                           for r in range(0, g[5], rows)]))
    return (out, torch.stack(stack)) if case["per_view"] else out


def _exact_points(case, seed):
    s = _kept(case, seed)
    dev = [[torch.from_numpy(a).to(DEVICE) for a in k] for k in s["keep"]]
    cos10 = float(np.float32(math.cos(math.radians(10.0))))

    def turn(R, n):                   # normals are 32-bit data, turned and compared in 32 bits
        R = torch.tensor(np.asarray(R, np.float32), device=DEVICE)
        return [(R[k, 0] * n[:, 0] + R[k, 1] * n[:, 1]) + R[k, 2] * n[:, 2] for k in range(3)]

    def project(P, X):
        w = P[2, 0] * X[0] + P[2, 1] * X[1] + P[2, 2] * X[2] + P[2, 3]
        return [(P[k, 0] * X[0] + P[k, 1] * X[1] + P[k, 2] * X[2] + P[k, 3]) / w for k in range(2)]

    xyz = []
    for i, (d, nrm, _) in enumerate(dev):
        v, u = torch.nonzero(d > 0, as_tuple=True)
        u64, v64 = u.double(), v.double()
        X = _back(s["inv"][i], u64, v64, d[v, u].double())
        n = turn(s["rot"][i], nrm[v, u])
        total = [x.clone() for x in X]
        count = torch.ones_like(u)
        first = torch.ones_like(u, dtype=torch.bool)
        for j, (dj, nj, _) in enumerate(dev):
            if j == i:
                continue
            p = project(s["P4"][j], X)
            cx, cy = torch.floor(p[0] + 0.5), torch.floor(p[1] + 0.5)
            ok = (cx >= 0) & (cy >= 0) & (cx < dj.shape[1]) & (cy < dj.shape[0])
            cx, cy = torch.where(ok, cx, 0 * cx), torch.where(ok, cy, 0 * cy)
            at = (cy.long(), cx.long())
            ok &= dj[at] > 0
            Y = _back(s["inv"][j], cx, cy, dj[at].double())
            ok &= sum((a - b) ** 2 for a, b in zip(Y, X)).sqrt() <= 1.0
            q = project(s["P4"][i], Y)
            ok &= ((q[0] - u64) ** 2 + (q[1] - v64) ** 2).sqrt() <= 2.0
            m = turn(s["rot"][j], nj[at])
            ok &= (n[0] * m[0] + n[1] * m[1]) + n[2] * m[2] >= cos10
            if j < i:
                first &= ~ok
            count += ok
            for k in range(3):
                total[k] += torch.where(ok, Y[k], torch.zeros_like(Y[k]))
        keep = first & (count >= 4)
        xyz.append(torch.stack([t[keep] / count[keep] for t in total]))
    xyz = torch.cat(xyz, 1)
    E, N, z = _utm(*xyz)
    dsm = _raster(E, N, z, s["grid"])
    return dict(points=xyz.shape[1], dsm=dsm, smooth=_blur(dsm))
