"""The work that users of this framework have it do, as cases to be timed.

Every case goes through the public entry points of doi_amd.rte on host arrays, as a
program calls them: optical maps and beams in, images (and gradients, Jacobians, fields)
out.  The sizes are those of the repository's own configurations (8^3 L=3, 16^3 L=5,
24^3 L=5, the 8-32^3 serving mix, the 32^3 L=5 batch), of its tests (ragged grids, the
other orders, the lambda stop rule, prop_thresh) and of the reference's published table
(20^3 L=3).  A pass starts from new optical maps: media, path tables and workspaces that
depend on them are made inside it, as for every step of a reconstruction or a data set.

Images of the mixed and FP32 precisions are kept as float32, the precision that their
propagation has; those of RTE_PREC_FP64 as float64.
"""
import math

import numpy as np
import torch

from doi_amd import rte

TERMS = 20        # Neumann terms of a solve to a 1e-6 relative change at these optics (17 to 22)
PREC = {"mixed": rte.PREC_MIXED, "fp64": rte.PREC_FP64, "fp32": rte.PREC_FP32}
C_LIGHT = 2.9979e10


def _case(name, kind, nx, ny, nz, L, g=0.9, media=1, beams=1, prec="mixed", path="cached", rule="delta",
          thresh=0.0, sigma=0.3, mus=1.0, n=1.0, blocks=0, omega=0.0):
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, L=L, g=g, media=media, beams=beams, prec=prec, path=path, rule=rule,
             thresh=thresh, sigma=sigma, mus=mus, n=n, blocks=blocks, omega=omega)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's plain solve: a small uniform cube, latency of one call
        _case("solve 8^3 L3 uniform", "solve", 8, 8, 8, 3, g=0.8, sigma=0.0, rule="lambda"),
        # one heterogeneous medium with its reflectance, the size of the oracle comparison
        _case("images 16^3 L5", "images", 16, 16, 16, 5, g=0.8, sigma=0.2),
        # one request at the size of the headline metric
        _case("solve 32^3 L5", "solve", 32, 32, 32, 5),
        # the headline batch (media x 5 beams at 32^3, L=5), with fewer media
        _case("batch 3x5 32^3 L5", "images", 32, 32, 32, 5, media=3, beams=5),
        # a low-order batch of a data set
        _case("batch 8x5 24^3 L3", "images", 24, 24, 24, 3, media=8, beams=5, sigma=0.2),
        # a phantom with its own proportions: ragged grid, cut-off couplings, the reference's stop rule
        _case("ragged 2x3 21x17x30 L4", "images", 21, 17, 30, 4, g=0.8, media=2, beams=3, rule="lambda", thresh=2.05,
              n=1.37),
        # the error reference that results are checked against, with the final radiance field
        _case("fp64 field 14^3 L5", "field", 14, 14, 14, 5, g=0.8, prec="fp64"),
        # the plain path: one solve, FP32, path integrals marched per pair (reference table: 20^3 L=3)
        _case("plain 20^3 L3 march", "solve", 20, 20, 20, 3, g=0.8, prec="fp32", path="march"),
        # frequency domain: modulated beams, phase images
        _case("fd 2x2 24^3 L5 100MHz", "fd", 24, 24, 24, 5, media=2, beams=2, omega=2 * math.pi * 1e8, sigma=0.2),
        # one step of a reconstruction: the loss and its gradient in every voxel
        _case("gradient 24^3 L5", "gradient", 24, 24, 24, 5, g=0.8, sigma=0.2),
        # the Fisher information's forward-mode Jacobian (4x4x4 blocks)
        _case("jacobian 64 blocks 20^3 L5", "jacobian", 20, 20, 20, 5, g=0.8, sigma=0.2, blocks=4),
        # a burst of the serving stream: mixed grids and orders submitted together
        _case("serve 24 requests 8-32^3", "serve", 32, 32, 32, 5, media=24),
    ]


def _cost(c):
    """Device work of a pass, relative: pair-coefficients of all its propagations."""
    N, K = c["nx"] * c["ny"] * c["nz"], (c["L"] + 1) ** 2
    per = {"images": 1, "solve": 1, "field": 1, "fd": 2.2, "gradient": 3, "jacobian": 1, "serve": 0.4}[c["kind"]]
    n = c["blocks"] ** 3 + 1 if c["kind"] == "jacobian" else c["media"] * c["beams"]
    slow = {"fp64": 8, "mixed": 1, "fp32": 1}[c["prec"]] * (10 if c["path"] == "march" else 1)
    return float(N) * N * (4 * K + 16) * per * n * slow + 2e9


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["solve", "images", "images", "images", "field", "fd", "gradient", "jacobian", "serve"])
        e = [int(round(6 * (32 / 6) ** rng.random())) for _ in range(3)]
        if rng.random() < 0.4 or kind == "serve":
            e = [e[0]] * 3
        prec = rng.choice(["mixed", "mixed", "mixed", "mixed", "fp64", "fp32"])
        if prec == "fp32" and kind in ("gradient", "jacobian", "field"):
            prec = "mixed"
        if kind == "serve":
            prec = "mixed"
        path = "march" if prec == "fp32" and kind == "solve" and rng.random() < 0.5 else "cached"
        many = kind in ("images", "fd")
        c = _case(None, kind, e[0], e[1], e[2], rng.choice([1, 2, 3, 3, 4, 5, 5, 5, 6, 7]),
                  g=round(rng.uniform(0.7, 0.9), 3), media=rng.randint(1, 4) if many else 1,
                  beams=rng.randint(1, 6) if many else 1, prec=prec, path=path,
                  rule=rng.choice(["delta", "delta", "lambda"]) if kind in ("images", "solve", "field") else "delta",
                  thresh=round(rng.uniform(1.0, 2.5), 3) if many and rng.random() < 0.2 else 0.0,
                  sigma=rng.choice([0.0, 0.2, 0.3]), mus=round(rng.uniform(0.5, 1.5), 3),
                  n=rng.choice([1.0, 1.37]), blocks=rng.randint(2, 3) if kind == "jacobian" else 0,
                  omega=2 * math.pi * 1e8 * rng.uniform(0.5, 5) if kind == "fd" else 0.0)
        if kind == "serve":
            c["media"] = rng.randint(8, 24)
            c["sigma"], c["mus"], c["n"] = 0.2, 1.0, 1.0
        if _cost(c) <= 0.6 * most:
            return c


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _bounds(nx, ny, nz, dx=0.1):
    return (-nx * dx / 2, nx * dx / 2, -ny * dx / 2, ny * dx / 2, 0.0, nz * dx)


def _maps(rng, nx, ny, nz, mua, mus, sigma):
    """Lognormal maps with one to three absorbing spheres; sigma 0: uniform with its levels."""
    N = nx * ny * nz
    if sigma == 0.0:
        f = rng.uniform(0.9, 1.1, 2)
        return np.full(N, mua * f[0]), np.full(N, mus * f[1])
    ma = mua * np.exp(sigma * rng.standard_normal(N))
    ms = mus * np.exp(sigma * rng.standard_normal(N))
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    for _ in range(rng.integers(1, 4)):
        c = [rng.uniform(0, e - 1) for e in (nx, ny, nz)]
        r = rng.uniform(2, 5)
        inside = ((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2 <= r * r).ravel()
        ma[inside] *= rng.uniform(1.5, 3.0)
    return ma, ms


def _beam(rng, nx, ny, dx=0.1):
    """One voxel column of the top face."""
    i, j = rng.integers(0, nx), rng.integers(0, ny)
    return (float((i + 0.5) * dx - nx * dx / 2), float((j + 0.5) * dx - ny * dx / 2), dx, 1.0)


def _params(c):
    return rte.make_params(c["L"], precision=PREC[c["prec"]],
                           stop_rule=rte.STOP_LAMBDA if c["rule"] == "lambda" else rte.STOP_DELTA, tol=1e-6,
                           max_terms=30, prop_thresh=c["thresh"],
                           path_mode=rte.PATH_MARCH if c["path"] == "march" else rte.PATH_CACHED)


def _inputs(case, seed):
    """Host arrays of a case, from the seed alone (run and exact both start here)."""
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, case["nx"], case["ny"], case["nz"], case["L"]])
    c = case
    shape = (c["nx"], c["ny"], c["nz"])
    if c["kind"] == "serve":
        # the serving stream's distribution; every fifth request has the largest edge
        edges = [e for e in (8, 12, 16, 24, 32) if e <= c["nx"]] or [c["nx"]]
        reqs = []
        for k in range(c["media"]):
            e, L = edges[k % len(edges)], (3, 5)[(k // len(edges)) % 2]
            ma, ms = _maps(rng, e, e, e, rng.uniform(0.005, 0.05), rng.uniform(0.5, 1.5), 0.2)
            reqs.append(dict(shape=(e, e, e), bounds=_bounds(e, e, e), mu_a=ma, mu_s=ms, L=L,
                             g=float(rng.uniform(0.7, 0.9)), beam=_beam(rng, e, e)))
        return dict(reqs=reqs)
    maps = [_maps(rng, *shape, 0.01, c["mus"], c["sigma"]) for _ in range(c["media"])]
    if c["rule"] == "lambda" and c["media"] == 1 and c["sigma"] == 0.0:
        beams = [(0.0, 0.0, 0.2, 1.0)]          # the plain solve's centred beam, several columns wide
        if c["nx"] % 2 or c["ny"] % 2:
            beams = [_beam(rng, c["nx"], c["ny"])]
    else:
        beams = [_beam(rng, c["nx"], c["ny"]) for _ in range(c["beams"])]
    d = dict(shape=shape, bounds=_bounds(*shape), maps=maps, beams=beams)
    if c["kind"] == "gradient":
        # the measured image: a smooth spot of the size of the solve's own exitance
        j, i = np.meshgrid(np.arange(c["ny"]), np.arange(c["nx"]), indexing="ij")
        s = rng.uniform(0.15, 0.3) * c["nx"]
        spot = np.exp(-((i - c["nx"] / 2) ** 2 + (j - c["ny"] / 2) ** 2) / (2 * s * s))
        d["target"] = rng.uniform(0.05, 0.15) * spot / spot.sum()
    if c["kind"] == "jacobian":
        b = c["blocks"]
        z, y, x = np.meshgrid(*[np.arange(e) for e in shape[::-1]], indexing="ij")
        d["part"] = ((x * b // c["nx"]) + b * ((y * b // c["ny"]) + b * (z * b // c["nz"]))).ravel().astype(np.int32)
    return d


_kept = {}


def _context():
    """The context that a program keeps for its lifetime."""
    if "ctx" not in _kept:
        _kept["ctx"] = rte.Context(0)
    return _kept["ctx"]


def _server():
    """The server that a serving program keeps for its lifetime (on a context of its own)."""
    if "server" not in _kept:
        _kept["server_ctx"] = rte.Context(0)
        _kept["server"] = rte.Server(_kept["server_ctx"], hbm_budget=48 << 30)
    return _kept["server"]


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = dict(case)
    if case["kind"] == "serve":
        s["server"] = _server()
        for r in s["reqs"]:
            r["params"] = rte.make_params(r["L"], precision=rte.PREC_MIXED, stop_rule=rte.STOP_DELTA, tol=1e-6,
                                          max_terms=30)
    else:
        s["ctx"] = _context()
        s["params"] = _params(case)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "serve":
        srv = s["server"]
        ids = [srv.submit(r["shape"], r["bounds"], r["mu_a"], r["mu_s"], r["g"], r["beam"], r["params"])
               for r in s["reqs"]]
        return [srv.wait(i)[1].astype(np.float32) for i in ids]
    kept = np.float64 if c["prec"] == "fp64" else np.float32
    ctx, p, shape, bounds = s["ctx"], s["params"], s["shape"], s["bounds"]
    if kind == "solve":
        ma, ms = s["maps"][0]
        img, _ = ctx.solve(shape, bounds, ma, ms, c["g"], s["beams"][0], p, n=c["n"])
        return img.astype(kept)
    media = [ctx.medium(shape, bounds, ma, ms, c["g"], c["n"]) for ma, ms in s["maps"]]
    try:
        if kind in ("images", "fd"):
            mm = [m for m in media for _ in s["beams"]]
            bb = list(s["beams"]) * len(media)
            if kind == "images":
                img, refl, _ = ctx.solve_images(mm, bb, p)
                return dict(trans=[x.astype(kept) for x in img], refl=refl.astype(kept))
            img, refl, _ = ctx.solve_fd(mm, bb, c["omega"], p)
            kc = np.complex128 if c["prec"] == "fp64" else np.complex64
            return dict(trans=[x.astype(kc) for x in img], refl=refl.astype(kc))
        if kind == "field":
            field, img, refl, _ = ctx.solve_field(media[0], s["beams"][0], p)
            return [x.astype(kept) for x in (field, img, refl)]
        if kind == "gradient":
            loss, img, ga, gs, _ = ctx.gradient(media[0], s["beams"][0], p, s["target"])
            return [x.astype(kept) for x in (np.array([loss]), img, ga, gs)]
        J, img, _ = ctx.ref_jacobian(media[0], s["beams"][0], p, s["part"], c["blocks"] ** 3)
        return [x.astype(kept) for x in (J, img)]
    finally:
        for m in media:
            m.close()


def work(case):
    """Maps in and images out once; the operations of the coupled pairs (projection onto and out of the
    SH basis per right-hand side, the pair's geometry once per medium) in the terms of a solve."""
    c = case

    def series(nx, ny, nz, L, media, rhs, terms, mult=1.0):
        N, K = nx * ny * nz, (L + 1) ** 2
        pairs = N * (N - 1.0)
        if c["thresh"] > 0:
            pairs *= min(1.0, 4.19 * (c["thresh"] / 0.1) ** 3 / N)
        return media * (16.0 * N + 16.0 * nx * ny * rhs), media * terms * pairs * (4.0 * K * rhs * mult + 16)

    if c["kind"] == "serve":
        b = f = 0.0
        for r in _inputs(case, 1)["reqs"]:
            x = series(*r["shape"], r["L"], 1, 1, TERMS)
            b, f = b + x[0], f + x[1]
        return {"bytes": b, "flops": f}
    g = (c["nx"], c["ny"], c["nz"])
    N, K = g[0] * g[1] * g[2], (c["L"] + 1) ** 2
    if c["kind"] == "jacobian":
        n = c["blocks"] ** 3
        b, f = series(*g, c["L"], 1, n + 1, TERMS)
        return {"bytes": b, "flops": f}
    mult = {"fd": 2.0, "gradient": 2.5}.get(c["kind"], 1.0)
    b, f = series(*g, c["L"], c["media"], c["beams"], TERMS, mult)
    extra = 8.0 * K * N if c["kind"] == "field" else 16.0 * N if c["kind"] == "gradient" else 0.0
    return {"bytes": b + extra, "flops": f}


# ---------------------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------
F64 = torch.float64
PAIRS = 1 << 23   # pairs of one piece


class _Medium:
    """Geometry, optics and the pair couplings kf = e^{-tau}/r^2 of one medium, [source, destination]."""

    def __init__(self, shape, bounds, ma, ms, g, L, n, thresh):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.shape, self.L, self.K, self.g, self.n, self.thresh = shape, L, (L + 1) ** 2, g, n, thresh
        nx, ny, nz = shape
        self.N, self.P = nx * ny * nz, nx * ny
        self.d = [(bounds[2 * i + 1] - bounds[2 * i]) / shape[i] for i in range(3)]
        self.dV = self.d[0] * self.d[1] * self.d[2]
        self.bounds = bounds
        v = torch.arange(self.N, device=self.dev)
        self.ijk = torch.stack([v % nx, (v // nx) % ny, v // (nx * ny)])
        self.ma = torch.tensor(ma, dtype=F64, device=self.dev)
        self.ms = torch.tensor(ms, dtype=F64, device=self.dev)
        self.mt = self.ma + self.ms
        self.step = max(1, PAIRS // self.N)
        self.mom = self._moments()
        self.kf = torch.empty(self.N, self.N, dtype=F64, device=self.dev)
        for s in range(0, self.N, self.step):
            tau, r2, off = self._march(s, lambda v, seg, acc: acc.add_(self.mt[v] * seg))
            k = torch.exp(-tau) / r2
            k[off] = 0.0
            self.kf[s:s + self.step] = k

    def _geometry(self, s):
        src = self.ijk[:, s:s + self.step]
        D = self.ijk[:, None, :] - src[:, :, None]
        x = [D[i].to(F64) * self.d[i] for i in range(3)]
        return src, D, x, x[0] ** 2 + x[1] ** 2 + x[2] ** 2

    def _march(self, s, visit):
        """Walks every ray of a piece of sources from voxel centre to voxel centre; visit(voxels, lengths, acc)."""
        nx, ny, _ = self.shape
        src, D, x, r2 = self._geometry(s)
        self_pair = (D == 0).all(0)
        r2 = torch.where(self_pair, 1.0, r2)
        r = r2.sqrt()
        n = D.abs()
        inc = [torch.where(n[i] > 0, 1.0 / n[i].clamp(min=1).to(F64), 1e30) for i in range(3)]
        a = [0.5 * t for t in inc]
        stride = [torch.where(D[i] > 0, m, -m) for i, m in enumerate((1, nx, nx * ny))]
        v = (src[0] + nx * (src[1] + ny * src[2]))[:, None].expand(-1, self.N).clone()
        left = n.sum(0)
        prev, acc = torch.zeros_like(r2), torch.zeros_like(r2)
        last = torch.zeros_like(r2)
        for t in range(int(left.max())):
            on = left > t
            pz = (a[2] <= a[0]) & (a[2] <= a[1])
            py = ~pz & (a[1] <= a[0])
            al = torch.where(pz, a[2], torch.where(py, a[1], a[0]))
            visit(v, torch.where(on, (al - prev) * r, 0.0), acc)
            prev = torch.where(on, al, prev)
            last = torch.where(on, torch.where(pz, inc[2], torch.where(py, inc[1], inc[0])), last)
            v = torch.where(on, v + torch.where(pz, stride[2], torch.where(py, stride[1], stride[0])), v)
            a = [torch.where(on & m, a[i] + inc[i], a[i]) for i, m in enumerate((~pz & ~py, py, pz))]
        visit(v, 0.5 * last * r, acc)
        off = self_pair
        if self.thresh > 0:
            off = off | (r2 >= self.thresh ** 2)
        return acc, r2, off

    def _harmonics(self, x, y, z):
        """Real orthonormal harmonics along the first axis, a = l^2 + l + m."""
        L = self.L
        out = [None] * self.K
        c, s = torch.ones_like(x), torch.zeros_like(x)
        for m in range(L + 1):
            if m:
                c, s = c * x - s * y, s * x + c * y
            p0, p1 = None, torch.full_like(z, float((-1) ** m * np.prod(np.arange(2 * m - 1, 0, -2))))
            for l in range(m, L + 1):
                if l > m:
                    p0, p1 = p1, ((2 * l - 1) * z * p1 - ((l + m - 1) * p0 if p0 is not None else 0.0)) / (l - m)
                f = math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - m) / math.factorial(l + m))
                if m:
                    out[l * l + l + m] = math.sqrt(2) * f * p1 * c
                    out[l * l + l - m] = math.sqrt(2) * f * p1 * s
                else:
                    out[l * l + l] = f * p1
        return out

    def _moments(self):
        """Angular moments of the self-voxel block on the reference's 200 x 200 grid, its centre-to-face
        distance in single precision, the last face that accepts a ray kept from direction to direction."""
        A = 200
        th, ph = np.meshgrid(np.arange(A) * math.pi / A, np.arange(A) * 2 * math.pi / A, indexing="ij")
        u = np.stack([np.cos(ph) * np.sin(th), np.sin(ph) * np.sin(th), np.cos(th)]).reshape(3, -1).astype(np.float32)
        hit = np.full((3, A * A), np.nan, dtype=np.float32)
        ud = u.astype(np.float64)
        for ax in range(3):
            for f in (1.0, -1.0):
                with np.errstate(divide="ignore", invalid="ignore"):
                    h = (f * ud / ud[ax]).astype(np.float32)
                h[ax] = f
                ok = (u[ax] != 0) & (np.abs(h) <= 1).all(0) & (u[ax] * h[ax] >= 0)
                hit = np.where(ok, h, hit)
        for w in np.flatnonzero(np.isnan(hit[0])):
            hit[:, w] = hit[:, w - 1] if w else 0.0
        beta = np.sqrt(sum(hit[i].astype(np.float64) ** 2 * (self.d[i] / 2.0) ** 2 for i in range(3)))
        t = lambda q: torch.tensor(q, dtype=F64, device=self.dev)  # noqa: E731
        st = np.sin(th).ravel()
        R = torch.stack(self._harmonics(t(np.cos(ph).ravel() * st), t(np.sin(ph).ravel() * st), t(np.cos(th).ravel())))
        return [(R * t(st * beta ** k)) @ R.T for k in range(1, 17)]

    def self_block(self, W, mu):
        """The self-voxel block on W [..., K, N] with (possibly complex) mu."""
        f = (math.pi / 200) * (2 * math.pi / 200) / self.dV
        out, coef = 0.0, torch.ones_like(mu)
        for k in range(16):
            if k:
                coef = coef * (-mu) / (k + 1)
            M = self.mom[k].to(W.dtype)
            out = out + coef * (M @ W)
        return f * out

    def piece(self, s):
        """Harmonics of the pair directions of one piece of sources, [sources, K, N]."""
        _, D, x, r2 = self._geometry(s)
        ri = 1.0 / torch.where(r2 == 0, 1.0, r2).sqrt()
        Z = torch.stack(self._harmonics(x[0] * ri, x[1] * ri, x[2] * ri), dim=1)
        return Z, r2

    def pairs(self, W, kim=0.0):
        """sum over sources of kf Z (Z . W) for W [B, K, N] real (kim: B = 2, real and imaginary half)."""
        out = torch.zeros_like(W)
        for s in range(0, self.N, self.step):
            Z, r2 = self.piece(s)
            P = torch.bmm(W[:, :, s:s + self.step].permute(2, 0, 1).contiguous(), Z)
            T = P * self.kf[s:s + self.step, None, :]
            if kim:
                r = r2.sqrt() * kim
                c, q = torch.cos(r), torch.sin(r)
                T = torch.stack([T[:, 0] * c + T[:, 1] * q, T[:, 1] * c - T[:, 0] * q], dim=1)
            for b in range(W.shape[0]):
                out[b] += (Z * T[:, b, None, :]).sum(0)
        return out

    def quadrature(self):
        """Weights of w_l0 in the exitance and the reflectance (100-point left sums)."""
        u = np.arange(100) / 100.0
        f = 2 * math.pi * self.d[0] * self.d[1] / math.sqrt(4 * math.pi)
        leg = [np.polynomial.legendre.Legendre.basis(l) for l in range(self.L + 1)]
        e = [f * math.sqrt(2 * l + 1) * float(np.sum(leg[l](u) * u / 100)) for l in range(self.L + 1)]
        r = [-f * math.sqrt(2 * l + 1) * float(np.sum(leg[l](u - 1) * (u - 1) / 100)) for l in range(self.L + 1)]
        return e, r

    def gl(self):
        return torch.tensor([self.g ** l for l in range(self.L + 1) for _ in range(2 * l + 1)], dtype=F64,
                            device=self.dev)[:, None]

    def source(self, beam, ma, ms, kim=0.0):
        """First-scatter source [K, N] and ballistic image [P]."""
        nx, ny, nz = self.shape
        b = self.bounds
        i, j = self.ijk[0, :self.P], self.ijk[1, :self.P]
        x = i.to(F64) * self.d[0] + b[0] + self.d[0] / 2
        y = j.to(F64) * self.d[1] + b[2] + self.d[1] / 2
        inside = ((x - beam[0]) ** 2 + (y - beam[1]) ** 2).sqrt() <= (beam[2] + 1e-16) / 2
        fact = beam[3] / float(inside.sum())
        mt = (ma + ms).reshape(nz, self.P)
        if kim:
            mt = mt + 1j * kim
        att = torch.exp(-mt * self.d[2])
        T = torch.cat([torch.ones_like(att[:1]), torch.cumprod(att, 0)])
        base = fact * ms.reshape(nz, self.P) / mt * T[:-1] * (1 - att) / self.dV * inside
        W = [torch.zeros_like(base.reshape(-1)) for _ in range(self.K)]
        for l in range(self.L + 1):
            W[l * l + l] = (self.g ** l * math.sqrt((2 * l + 1) / (4 * math.pi)) * base).reshape(-1)
        return torch.stack(W), fact * T[-1] * inside


def _series(M, W, E, c, apply, mu, ms, kim=0.0, keep=None):
    """The Neumann series from first term W [K, N] and image E [P]: (image, reflectance, sum of A W)."""
    eq, rq = M.quadrature()
    a0 = [l * l + l for l in range(M.L + 1)]
    eq, rq = (torch.tensor(q, dtype=W.dtype, device=M.dev) for q in (eq, rq))
    ws = torch.zeros(M.K, dtype=F64, device=M.dev)
    for l in range(M.L + 1):
        ws[l * l + l] = 1.0
        for m in range(2, l + 1, 2):
            ws[l * l + l + m] = math.sqrt(2)
    R, phi = torch.zeros_like(E), 0.0
    lam = c["rule"] == "lambda"
    bottom = lambda w: float((ws @ w[:, -M.P:].detach().real).sum())  # noqa: E731
    total, n, out, fi, state = E.detach().sum(), int(lam), bottom(W), 1.0, 0
    while True:
        AW = M.dV * (apply(W) + M.self_block(W, mu))
        phi = phi + AW
        dE = eq @ AW[a0][:, -M.P:]
        E, R = E + dE, R + rq @ AW[a0][:, :M.P]
        total = total + dE.detach().sum()
        if state == 2:
            break
        n += 1
        W = M.gl().to(W.dtype) * ms * AW
        if not lam:
            if abs(complex(dE.detach().sum())) < 1e-6 * abs(complex(total)) or n >= 30:
                break
            continue
        s = bottom(W)
        out += s
        gam = s / out
        hi = 1.0 - gam / (1.0 - gam / fi)
        fi = gam
        if (0.0 <= hi <= 1.0 and hi > 0.9999) or n >= 30:
            state = 2
    return E, R, phi


def _cw(M, beam, c):
    W, ball = M.source(beam, M.ma, M.ms)
    return _series(M, W, ball, c, lambda w: M.pairs(w[None])[0], M.mt, M.ms)


def _fd(M, beam, c):
    kim = c["omega"] * c["n"] / C_LIGHT
    W, ball = M.source(beam, M.ma, M.ms, kim)

    def apply(w):
        p = M.pairs(torch.stack([w.real, w.imag]), kim)
        return torch.complex(p[0], p[1])
    return _series(M, W, ball, c, apply, M.mt + 1j * kim, M.ms)


class _Coupled(torch.autograd.Function):
    """M.pairs with its transpose, and the pair weights d/d tau summed into M.pair_grad."""

    @staticmethod
    def forward(ctx, W, M):
        ctx.M = M
        ctx.save_for_backward(W)
        return M.pairs(W[None])[0]

    @staticmethod
    def backward(ctx, G):
        M, (W,) = ctx.M, ctx.saved_tensors
        out = torch.zeros_like(W)
        for s in range(0, M.N, M.step):
            Z, _ = M.piece(s)
            k = M.kf[s:s + M.step]
            Q = k * (Z * G).sum(1)
            P = torch.bmm(W[:, s:s + M.step].T.contiguous()[:, None, :], Z)[:, 0]
            M.pair_grad[s:s + M.step] -= Q * P
            out[:, s:s + M.step] = (Z * Q[:, None, :]).sum(2).T
        return out, None


def _gradient(M, beam, c, target):
    M.pair_grad = torch.zeros_like(M.kf)
    ma, ms = M.ma.clone().requires_grad_(), M.ms.clone().requires_grad_()
    W, ball = M.source(beam, ma, ms)
    E, _, _ = _series(M, W, ball, c, lambda w: _Coupled.apply(w, M), ma + ms, ms)
    loss = ((E - torch.tensor(target.ravel(), dtype=F64, device=M.dev)) ** 2).sum()
    loss.backward()
    gt = torch.zeros(M.N, dtype=F64, device=M.dev)
    for s in range(0, M.N, M.step):
        w = M.pair_grad[s:s + M.step]
        M._march(s, lambda v, seg, acc: gt.index_add_(0, v.reshape(-1), (w * seg).reshape(-1)))
    return [loss.detach().reshape(1), E.detach().reshape(c["ny"], c["nx"]), ma.grad + gt, ms.grad + gt]


def _jacobian(M, beam, c, part):
    E, _, phi = _cw(M, beam, c)
    part = torch.tensor(part, device=M.dev)
    cols = []
    for a in range(c["blocks"] ** 3):
        W = -M.n * phi * (part == a)
        e, _, _ = _series(M, W, torch.zeros_like(E), c, lambda w: M.pairs(w[None])[0], M.mt, M.ms)
        cols.append(e)
    return [torch.stack(cols, 1), E.reshape(c["ny"], c["nx"])]


def _seconds(N, L, series, rhs=1):
    """About what a series of 20 terms takes here: the couplings once, then the terms."""
    return 9.0 * (N / 32768.0) ** 2 + series * rhs * 9.0 * (N / 32768.0) ** 2 * (L + 1) ** 2 / 36.0


def exact(case, seed):
    c = case
    s = _inputs(case, seed)
    host = lambda t: t.cpu().numpy()  # noqa: E731
    if c["kind"] == "serve":
        out, spent = [], 0.0
        for r in s["reqs"]:
            t = _seconds(int(np.prod(r["shape"])), r["L"], 1) + 0.4
            if spent + t > 16 or r["shape"][0] > 16:
                out.append(None)
                continue
            spent += t
            M = _Medium(r["shape"], r["bounds"], r["mu_a"], r["mu_s"], r["g"], r["L"], 1.0, 0.0)
            out.append(host(_cw(M, r["beam"], dict(rule="delta"))[0].reshape(r["shape"][1], r["shape"][0])))
        return out
    N = c["nx"] * c["ny"] * c["nz"]
    series = {"gradient": 4, "fd": 2}.get(c["kind"], c["blocks"] ** 3 + 1 if c["kind"] == "jacobian" else 1)
    image_only = c["kind"] == "jacobian" and _seconds(N, c["L"], series) > 19
    if _seconds(N, c["L"], 1 if image_only else series) > 19:
        return None
    medium = lambda k: _Medium(s["shape"], s["bounds"], *s["maps"][k], c["g"], c["L"], c["n"], c["thresh"])  # noqa: E731
    ny, nx = c["ny"], c["nx"]
    if c["kind"] == "solve":
        return host(_cw(medium(0), s["beams"][0], c)[0].reshape(ny, nx))
    if c["kind"] in ("images", "fd"):
        # as many of the batch's solves as the time allows, the first ones
        one = _cw if c["kind"] == "images" else _fd
        trans, refl, spent = [], [], 0.0
        for k in range(c["media"]):
            M = None
            for b in s["beams"]:
                spent += _seconds(N, c["L"], series) * (1.0 if M is None else 0.6)
                if spent > 19:
                    trans.append(None)
                    refl.append(None)
                    continue
                M = M or medium(k)
                E, R, _ = one(M, b, c)
                trans.append(host(E.reshape(ny, nx)))
                refl.append(host(R.reshape(ny, nx)))
        whole = None if any(r is None for r in refl) else np.stack(refl)
        return dict(trans=trans, refl=whole)
    M = medium(0)
    if c["kind"] == "field":
        E, R, phi = _cw(M, s["beams"][0], c)
        return [host(phi * (c["n"] / C_LIGHT)), host(E.reshape(ny, nx)), host(R.reshape(ny, nx))]
    if c["kind"] == "gradient":
        return [host(t) for t in _gradient(M, s["beams"][0], c, s["target"])]
    if image_only:
        return [None, host(_cw(M, s["beams"][0], c)[0].reshape(ny, nx))]
    return [host(t) for t in _jacobian(M, s["beams"][0], c, s["part"])]
