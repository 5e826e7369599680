"""The work a user of this framework has it do, as measurable cases.

A host program advances a colony of rod cells in one or many traps.  Per time
step it hands the cells over (sample every species at every cell, deposit what
the cells make), has the field step solved and takes the fields or the samples
back.  Every case is one such time step through the public binding
(`eq_amd.field`), from the reference's 160 x 80 trap fed from host arrays to
four species on an 8192 x 4096 trap with flow and a batch of hundreds of
uneven traps.

A case's plain values: grid (`nx`, `ny` cells, `npm` nodes per micron),
`species`, `rods` (per trap), `walls`, solver `kind`, `mode`:
  dev      cells and fields stay on the device (couple_dev, step, download_dev)
  host     cells, samples and fields in host arrays (couple, step, download)
  vectors  no cells: the solution vector goes in and out of every solve
  affine   amounts that depend on the cell's own sample (couple_affine_dev)
  tensor   the diffusion tensor follows the cells' angles (EQ_COUPLE_TENSOR)
  channels flow channels above and below the trap
  well     a boundary well on four Dirichlet walls
  flow     a prescribed channel velocity (nonsymmetric: BiCGStab)
  traps    `traps` uneven traps in one batch
"""
import math
import random

import numpy as np
import torch

from eq_amd import field as F

DT = 0.1
KINDS = {"mixed": F.MIXED_GMG_CG, "gmg": F.GMG_CG, "ir": F.IR_GMG_CG, "mixed_bicgstab": F.MIXED_GMG_BICGSTAB,
         "gmg_bicgstab": F.GMG_BICGSTAB}
# which walls are held (value 0) or open at a Robin rate; the others are closed
WALLS = {"top": {F.TOP: "D"}, "bottom": {F.BOTTOM: "D"}, "all": {w: "D" for w in range(4)},
         "channels": {F.TOP: "D", F.BOTTOM: "D"}, "closed": {},
         "sides": {F.TOP: "D", F.LEFT: "R", F.RIGHT: "R"}}
ROBIN_RATE, ROBIN_S = 1.5, 0.2
TENSOR = (1.0, 0.5)     # axial and transverse diffusion along a rod
EXCHANGE = -0.05        # membrane exchange: q = a + EXCHANGE * (the cell's own sample)
POSITIONS = 4           # cell positions of successive steps, in hand before the call


def case(name, nx, ny, npm, rods, mode="dev", kind="mixed", walls="top", species=2, traps=1, scheme="p1", layout=0):
    return {"name": name, "nx": nx, "ny": ny, "npm": npm, "rods": rods, "mode": mode, "kind": kind, "walls": walls,
            "species": species, "traps": traps, "scheme": scheme, "layout": layout}


def listed():
    return [
        # the reference's own set-up: every array on the host, a step as short as its launches
        case("reference trap, host arrays", 160, 80, 4, 200, mode="host"),
        # the finite-difference solver's use: solution vector in, solve, solution vector out
        case("fd vectors 400x200", 400, 200, 10, 0, mode="vectors", kind="gmg", scheme="fd"),
        # a microfluidic trap open to flow channels on two sides
        case("channels 437x221", 437, 221, 10, 600, mode="channels", walls="channels"),
        # diffusion along the rods' axes
        case("cell tensor 800x400", 800, 400, 10, 2000, mode="tensor"),
        # strains whose production follows their own reading
        case("affine coupling 1000x500", 1000, 500, 20, 1000, mode="affine"),
        # a trap whose sizes divide by nothing
        case("odd trap 1237x611", 1237, 611, 20, 1500),
        # production: one large trap, 5000 walking rods
        case("trap 2000x1000", 2000, 1000, 20, 5000),
        # the same solved in FP64 throughout
        case("trap 2000x1000 fp64", 2000, 1000, 20, 5000, kind="gmg"),
        # a parameter scan's batch: a few uneven traps, and hundreds
        case("12 uneven traps", 0, 0, 10, 0, mode="traps", traps=12, layout=1),
        case("512 uneven traps", 0, 0, 10, 0, mode="traps", traps=512, layout=3),
        # flow through the trap, ordinary and large
        case("flow 901x449", 901, 449, 20, 900, mode="flow", kind="mixed_bicgstab"),
        case("flow 8192x4096, 4 species", 8192, 4096, 40, 100000, mode="flow", kind="mixed_bicgstab", species=4),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: sizes spread over their logarithm, odd ones among them."""
    mode = rng.choices(["dev", "traps", "host", "channels", "tensor", "affine", "flow", "vectors", "well"],
                       [10, 4, 2, 2, 2, 2, 3, 2, 1])[0]
    kind = rng.choices(["mixed", "gmg", "ir"], [7, 3, 1])[0]
    species = rng.choice([1, 2, 2, 2, 3, 4])
    npm = rng.choice([4, 10, 10, 20])
    lo, hi = {"dev": (150, 3000), "host": (100, 800), "affine": (100, 1200), "tensor": (150, 1600), "flow": (150, 3000),
              "channels": (100, 1500), "vectors": (100, 1600), "well": (100, 1500), "traps": (0, 0)}[mode]
    if mode == "traps":
        return _unnamed(case("", 0, 0, 10, 0, mode="traps", kind="mixed", traps=int(_log(rng, 2, 200)),
                             layout=rng.randrange(4, 1 << 20)))
    nx = int(_log(rng, lo, hi))
    ny = max(40, int(nx * rng.uniform(0.3, 1.0)))
    rods = 0 if mode in ("vectors", "well") else max(5, int(nx / npm * ny / npm * rng.uniform(0.2, 1.0)))
    if mode == "affine":
        rods = min(rods, 2000)
    scheme = rng.choice(["p1", "fd"]) if mode == "vectors" else "p1"
    walls = {"channels": "channels", "well": "all"}.get(mode) or rng.choice(["top", "top", "top", "bottom", "all", "sides"])
    if mode == "flow":
        kind = rng.choice(["mixed_bicgstab", "mixed_bicgstab", "gmg_bicgstab"])
    if mode in ("channels", "well"):
        kind = rng.choice(["mixed", "gmg"])
    return _unnamed(case("", nx, ny, npm, rods, mode=mode, kind=kind, walls=walls, species=species, scheme=scheme))


def _unnamed(c):
    del c["name"]
    return c


class _Trap:
    """One trap's grid and species: the same for every seed."""

    def __init__(self, nx, ny, npm, rods, D, gamma):
        self.nx, self.ny, self.npm, self.rods, self.D, self.gamma = nx, ny, float(npm), rods, D, gamma
        self.width, self.height = nx / npm, ny / npm
        self.n = (nx + 1) * (ny + 1)


def _traps(c):
    rng = random.Random(c["layout"])
    if c["mode"] != "traps":
        D = [400.0, 100.0] if c["species"] == 2 else [400.0, 250.0, 150.0, 100.0][: c["species"]]
        return [_Trap(c["nx"], c["ny"], c["npm"], c["rods"], D, [0.01] * c["species"])]
    out = []
    for _ in range(c["traps"]):  # 20-100 um by 10-50 um, 50-3000 rods, each with its own rates
        nx, ny = rng.randint(200, 1000), rng.randint(100, 500)
        g = 10.0 ** rng.uniform(-3.0, -1.0)
        out.append(_Trap(nx, ny, c["npm"], rng.randint(50, 3000),
                         [rng.uniform(200.0, 600.0), rng.uniform(50.0, 150.0)], [g, g]))
    return out


def _walls(c):
    return {w: (F.DIRICHLET, 0.0, 0.0, 0.0) if k == "D" else (F.ROBIN, 0.0, ROBIN_RATE, ROBIN_S)
            for w, k in WALLS[c["walls"]].items()}


def _cells(c, traps, seed):
    """Per trap: rods at POSITIONS successive steps of a random walk, (POSITIONS, rods, 5), and their amounts per step."""
    rng = np.random.default_rng([seed, 1])
    cells, q = [], []
    for t in traps:
        k = t.rods
        a = np.empty((POSITIONS, k, 5))
        lim = np.array([t.width, t.height])
        a[0, :, :2] = rng.random((k, 2)) * lim
        a[0, :, 2] = rng.random(k) * math.pi
        a[0, :, 3] = rng.uniform(2.0, 4.0, k)
        a[0, :, 4] = 1.0
        for s in range(1, POSITIONS):
            a[s] = a[s - 1]
            a[s, :, :2] = np.clip(a[s, :, :2] + 0.05 * rng.standard_normal((k, 2)), 0.0, lim)
        cells.append(a)
        q.append(rng.uniform(0.5, 1.5, (k, c["species"])) * DT)
    return cells, q


def _fields(c, traps, seed, device):
    """Per problem: the smooth concentration of a run under way, zero on held walls, (ny+1, nx+1)."""
    rng = np.random.default_rng([seed, 2])
    held = [w for w, k in WALLS[c["walls"]].items() if k == "D"]
    out = []
    for t in traps:
        x = torch.linspace(0.0, 1.0, t.nx + 1, dtype=torch.float64, device=device)[None, :]
        y = torch.linspace(0.0, 1.0, t.ny + 1, dtype=torch.float64, device=device)[:, None]
        wall = torch.ones_like(x * y)
        for w in held:
            far = (x, 1.0 - x, 1.0 - y, y)[w]
            wall = wall * torch.sin(0.5 * math.pi * far) if len(held) < 4 else wall * (1.0 - (1.0 - far) ** 8)
        for _ in range(c["species"]):
            u = torch.ones_like(wall)
            for kx, ky in ((1, 0), (0, 2), (2, 1), (5, 3)):
                u = u + 0.15 * float(rng.uniform(-1, 1)) * torch.cos(math.pi * kx * x) * torch.cos(math.pi * ky * y)
            out.append(0.02 * u * wall)
    return out


def _velocity(t):
    y = np.arange(t.ny + 1) * (t.height / t.ny)
    return 4.0 * 50.0 * y * (t.height - y) / (t.height * t.height)


def prepare(case, seed):
    c = case
    traps = _traps(c)
    ns = c["species"]
    walls = _walls(c)
    scheme = F.SCHEME_FD if c["scheme"] == "fd" else F.SCHEME_P1
    descs = [F.field_desc(t.nx, t.ny, t.width, t.height, DT, D, g, 0.0, walls, scheme=scheme)
             for t in traps for D, g in zip(t.D, t.gamma)]
    torch.cuda.current_stream().synchronize()
    fb = F.FieldBatch(descs, nspecies=ns, solver=F.solver_desc(KINDS[c["kind"]]))
    s = {"fb": fb, "case": c, "k": 0, "npm": float(c["npm"])}
    t0 = traps[0]
    for p in range(len(descs)):
        if c["mode"] == "flow":
            fb.set_velocity(p, _velocity(t0))
        if c["mode"] == "channels":
            D = t0.D[p]
            ends = (D / 5.0, 0.0, D / 7.0, 0.0, 2.0 * 10.0 * 3.0 * (t0.width + t0.height))
            fb.set_channels(p, F.channel_desc(20.0, *ends, 3), F.channel_desc(0.0, *ends, 1))
        if c["mode"] == "well":
            fb.set_well(p, 2.0 * 10.0 * 3.0 * (t0.width + t0.height), 0.5, 0.05)
    if c["mode"] == "tensor":
        fb.cell_tensor(0, *TENSOR)
    fields = _fields(c, traps, seed, "cuda")
    cells, q = _cells(c, traps, seed)
    if c["mode"] in ("host", "vectors"):
        s["u"] = [u.cpu().numpy().reshape(-1) for u in fields]
        s["cells"], s["q"] = cells[0], q[0]
        for p, u in enumerate(s["u"]):
            fb.upload(p, u)
        return s
    torch.cuda.synchronize()
    for p, u in enumerate(fields):
        fb.upload_dev(p, u.data_ptr(), u.numel())
    fb.sync()
    rods = sum(t.rods for t in traps)
    s["off"] = np.concatenate([[0], np.cumsum([t.rods for t in traps])]).astype(np.int64)
    s["cells"] = torch.from_numpy(np.concatenate(cells, axis=1)).cuda().contiguous()
    s["q"] = torch.from_numpy(np.concatenate(q)).cuda().contiguous()
    s["b"] = torch.full_like(s["q"], EXCHANGE)
    s["sampled"] = torch.zeros((rods, ns), dtype=torch.float64, device="cuda")
    s["counts"] = torch.zeros(rods, dtype=torch.int32, device="cuda")
    s["sizes"] = [u.numel() for u in fields]
    s["out"] = torch.zeros(sum(s["sizes"]), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    return s


def run(state):
    """One time step: cells to field, solve, and the fields and samples back."""
    s, c = state, state["case"]
    fb, mode = s["fb"], c["mode"]
    if mode == "vectors":
        for p, u in enumerate(s["u"]):
            fb.upload(p, u)
        fb.step()
        s["u"] = [fb.download(p) for p in range(len(s["u"]))]
        return {"fields": np.concatenate(s["u"])}
    k = s["k"] % POSITIONS
    s["k"] += 1
    if mode == "host":
        sampled, counts = fb.couple(0, s["cells"][k], s["npm"], s["q"])
        fb.step()
        return {"fields": np.concatenate([fb.download(p) for p in range(c["species"])]), "sampled": sampled,
                "counts": counts}
    cells = s["cells"][k]
    flags = F.SAMPLE | F.DEPOSIT | (F.TENSOR if mode == "tensor" else 0)
    if mode == "affine":
        fb.couple_affine_dev(0, s["off"], cells.data_ptr(), s["npm"], s["q"].data_ptr(), s["b"].data_ptr(),
                             s["sampled"].data_ptr(), s["counts"].data_ptr())
    elif mode == "traps":
        fb.couple_traps_dev(0, s["off"], cells.data_ptr(), s["npm"], s["q"].data_ptr(), s["sampled"].data_ptr(),
                            s["counts"].data_ptr(), flags)
    elif mode != "well":
        fb.couple_dev(0, cells.data_ptr(), cells.shape[0], s["npm"], s["q"].data_ptr(), s["sampled"].data_ptr(),
                      s["counts"].data_ptr(), flags)
    fb.step()
    at = s["out"].data_ptr()
    for p, n in enumerate(s["sizes"]):
        fb.download_dev(p, at, n)
        at += 8 * n
    got = {"fields": s["out"]}
    if mode == "well":
        got["wells"] = np.array([fb.well_state(p)[:2] for p in range(c["species"])])
        return got
    got["sampled"], got["counts"] = s["sampled"], s["counts"]
    if mode == "channels":
        got["channels"] = np.array([fb.channel_values(p) for p in range(c["species"])])
    return got


def work(case):
    """Each field read and written once, each cell's record and amounts read, its samples and count written; per node a
    right-hand side row and one application of the operator (7 points each)."""
    traps, ns = _traps(case), case["species"]
    nodes = sum(t.n for t in traps) * ns
    rods = sum(t.rods for t in traps)
    covered = 3.0 * case["npm"] ** 2 * rods * ns
    return {"bytes": 16.0 * nodes + rods * (44.0 + 16.0 * ns), "flops": 34.0 * nodes + 2.0 * covered}


# ---------------------------------------------------------------- the same step in plain torch and numpy, 64 bits

def _index(v, npm):
    r = math.floor(v * npm + 0.5)
    return r if r > 0 else 0


def _covered(t, cell):
    """(row window, column window, mask) of the nodes strictly inside the rod's box, searched in the window around its
    poles; the centre node where there is none."""
    x, y, a, length, width = (float(v) for v in cell)
    cs, sn = math.cos(a), math.sin(a)
    edge = _index(0.5, t.npm)
    rows, cols = [], []
    for side in (1.0, -1.0):
        off = side * 0.5 * length - width / 2.0
        cols.append(_index(min(max(x + cs * off, 0.0), t.width), t.npm))
        rows.append(_index(min(max(y + sn * off, 0.0), t.height), t.npm))
    i1, i2 = max(min(rows) - edge, 0), min(max(rows) + edge, t.ny)
    j1, j2 = max(min(cols) - edge, 0), min(max(cols) + edge, t.nx)
    dx = np.arange(j1, j2 + 1)[None, :] / t.npm - x
    dy = np.arange(i1, i2 + 1)[:, None] / t.npm - y
    mask = (np.abs(cs * dx + sn * dy) < (length - width) / 2.0) & (np.abs(cs * dy - sn * dx) < width / 2.0)
    if not mask.any():
        i, j = min(_index(y, t.npm), t.ny), min(_index(x, t.npm), t.nx)
        return slice(i, i + 1), slice(j, j + 1), np.ones((1, 1), bool)
    return slice(i1, i2 + 1), slice(j1, j2 + 1), mask


def _couple_exact(t, cells, q, fields, exchange=0.0, tensor=None):
    """Cells in list order: each reads its mean, then adds its amount; fields (species, ny+1, nx+1) change in place."""
    sampled = np.empty_like(q)
    grids = None
    if tensor is not None:
        grids = [np.ones(fields.shape[1:]), np.ones(fields.shape[1:]), np.zeros(fields.shape[1:])]
    for k in range(cells.shape[0]):
        i, j, mask = _covered(t, cells[k])
        n = float(mask.sum())
        view = fields[:, i, j]
        sampled[k] = (view * mask).sum(axis=(1, 2)) / n
        view += ((q[k] + exchange * sampled[k]) / n)[:, None, None] * mask
        if grids is not None:
            cs, sn = math.cos(cells[k, 2]), math.sin(cells[k, 2])
            for g, v in zip(grids, (tensor[0] * cs * cs + tensor[1] * sn * sn, tensor[0] * sn * sn + tensor[1] * cs * cs,
                                    (tensor[0] - tensor[1]) * sn * cs)):
                g[i, j][mask] = v
    return sampled, grids


class _System:
    """(1 + dt gamma) M + dt K (+ Robin, + convection) on the grid, as seven-point rows; K in difference form."""

    def __init__(self, c, t, D, gamma, tensor, velocity, device):
        self.shape = (t.ny + 1, t.nx + 1)
        self.device = device
        hx, hy = t.width / t.nx, t.height / t.ny
        z = lambda: torch.zeros(self.shape, dtype=torch.float64, device=device)  # noqa: E731
        self.mass, self.stiff = {(0, 0): z()}, {}
        ones = z() + 1.0
        if c["scheme"] == "fd":
            w = ones.clone()
            for edge in (w[0], w[-1], w[:, 0], w[:, -1]):
                edge *= 0.5
            self.mass[(0, 0)] += w * hx * hy
            kx, ky = ones[:, 1:] * DT * D * hy / hx, ones[1:] * DT * D * hx / hy
            for edge in (kx[0], kx[-1], ky[:, 0], ky[:, -1]):
                edge *= 0.5
            self._pair(self.stiff, (0, 1), kx)
            self._pair(self.stiff, (1, 0), ky)
        else:
            d = [torch.from_numpy(g).to(device) for g in tensor] if tensor else [ones, ones, ones * 0.0]
            v = torch.from_numpy(velocity).to(device)[:, None] * ones if velocity is not None else None
            area = hx * hy / 2.0
            # vertices (di, dj) and gradients of the lower and upper triangle of every cell
            for tri, grad in ((((0, 0), (0, 1), (1, 1)), ((-1 / hx, 0.0), (1 / hx, -1 / hy), (0.0, 1 / hy))),
                              (((0, 0), (1, 0), (1, 1)), ((0.0, -1 / hy), (-1 / hx, 1 / hy), (1 / hx, 0.0)))):
                at = lambda a, p: a[p[0]:self.shape[0] - 1 + p[0], p[1]:self.shape[1] - 1 + p[1]]  # noqa: E731
                mean = [sum(at(g, p) for p in tri) / 3.0 for g in d]
                for pa, ga in zip(tri, grad):
                    for pb, gb in zip(tri, grad):
                        off = (pb[0] - pa[0], pb[1] - pa[1])
                        m = self.mass.setdefault(off, z())
                        at(m, pa).add_(area / 6.0 if pa == pb else area / 12.0)
                        if pa == pb:
                            continue
                        k = self.stiff.setdefault(off, z())
                        at(k, pa).add_(DT * D * area * (mean[0] * (ga[0] * gb[0]) + mean[1] * (ga[1] * gb[1]) +
                                                        mean[2] * (ga[0] * gb[1] + ga[1] * gb[0])))
                        if v is not None:
                            at(k, pa).add_(DT * gb[0] * area / 12.0 * (sum(at(v, p) for p in tri) + at(v, pa)))
        self.mass0 = {o: m.clone() for o, m in self.mass.items()}
        for m in self.mass.values():
            m *= 1.0 + DT * gamma
        self.source = z()
        self.free = ones
        for w, kind in WALLS[c["walls"]].items():
            at = {F.LEFT: (slice(None), 0), F.RIGHT: (slice(None), -1), F.TOP: (-1, slice(None)),
                  F.BOTTOM: (0, slice(None))}[w]
            if kind == "D":
                self.free[at] = 0.0
                continue
            e, step = (hy, (1, 0)) if w in (F.LEFT, F.RIGHT) else (hx, (0, 1))
            r = DT * ROBIN_RATE * e
            line = lambda a, lo, hi: a[at][lo:a[at].shape[0] + hi]  # noqa: E731
            fd = c["scheme"] == "fd"  # lumped there
            for lo, hi, off in ((0, -1, step), (1, 0, (-step[0], -step[1]))):
                line(self.mass[(0, 0)], lo, hi).add_(r / 2.0 if fd else r / 3.0)
                if not fd:
                    line(self.mass.setdefault(off, z()), lo, hi).add_(r / 6.0)
                line(self.source, lo, hi).add_(r * ROBIN_S / 2.0)

    def _pair(self, table, off, k):
        a = torch.zeros(self.shape, dtype=torch.float64, device=self.device)
        b = torch.zeros_like(a)
        n0, n1 = k.shape
        a[:n0, :n1] -= k
        b[off[0]:, off[1]:] -= k
        table[off], table[(-off[0], -off[1])] = a, b

    def _moved(self, x, off):
        y = torch.zeros_like(x)
        n0, n1 = self.shape
        a0, a1 = max(0, -off[0]), max(0, -off[1])
        b0, b1 = n0 - max(0, off[0]), n1 - max(0, off[1])
        y[a0:b0, a1:b1] = x[a0 + off[0]:b0 + off[0], a1 + off[1]:b1 + off[1]]
        return y

    def times(self, x):
        offs = set(self.mass) | set(self.stiff)
        moved = {o: x if o == (0, 0) else self._moved(x, o) for o in offs}
        y = sum(m * moved[o] for o, m in self.mass.items())
        for o, k in self.stiff.items():
            y += k * (moved[o] - x)
        return y

    def solve(self, u, symmetric):
        """The new field from `u` (held walls at 0), by Jacobi-preconditioned CG or BiCGStab, restarted on its true
        residual until that stops falling."""
        b = sum(m * (u if o == (0, 0) else self._moved(u, o)) for o, m in self.mass0.items()) + self.source
        b = b * self.free
        inv = self.free / (self.mass[(0, 0)] - sum(self.stiff.values()))
        x, best = u * self.free, None
        for _ in range(6):
            r = (b - self.times(x)) * self.free
            rel = float(r.norm() / b.norm()) if float(b.norm()) else 0.0
            if rel < 1e-14 or (best is not None and rel > 0.5 * best):
                break
            best = rel
            x = x + (self._cg if symmetric else self._bicgstab)(r, inv, 1e-14 * float(b.norm()))
        return x

    def _cg(self, r, inv, stop, most=20000):
        x, z = torch.zeros_like(r), r * inv
        p, rz = z.clone(), (r * z).sum()
        for k in range(most):
            q = self.times(p) * self.free
            a = rz / (p * q).sum()
            x.add_(a * p)
            r = r - a * q
            z = r * inv
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
            if k % 100 == 99 and not float(r.norm()) > stop:
                break
        return x

    def _bicgstab(self, r, inv, stop, most=6000):
        x, hat, p, v = torch.zeros_like(r), r.clone(), torch.zeros_like(r), torch.zeros_like(r)
        rho = alpha = omega = torch.ones((), dtype=torch.float64, device=r.device)
        for k in range(most):
            new = (hat * r).sum()
            p = r + (new / rho) * (alpha / omega) * (p - omega * v)
            rho = new
            y = p * inv
            v = self.times(y) * self.free
            alpha = rho / (hat * v).sum()
            s = r - alpha * v
            z = s * inv
            t = self.times(z) * self.free
            omega = (t * s).sum() / (t * t).sum()
            x = x + alpha * y + omega * z
            r = s - omega * t
            if k % 50 == 49 and not float(r.norm()) > stop:
                break
        return x


def exact(case, seed):
    c = case
    traps = _traps(c)
    if sum(t.n for t in traps) * c["species"] > 9_000_000 or sum(t.rods for t in traps) > 25_000 or len(traps) > 16 or \
            c["mode"] == "well" or (c["mode"] == "flow" and traps[0].n > 600_000):
        return None  # over 20 seconds (a well's wall value: its own first-step state)
    device = "cuda" if torch.cuda.is_available() else "cpu"
    fields = _fields(c, traps, seed, "cpu" if device == "cpu" else "cuda")
    cells, q = _cells(c, traps, seed)
    new, sampled = [], []
    for k, t in enumerate(traps):
        u = np.stack([f.cpu().numpy() for f in fields[k * c["species"]:(k + 1) * c["species"]]])
        got, tensor = _couple_exact(t, cells[k][0], q[k], u, EXCHANGE if c["mode"] == "affine" else 0.0,
                                    TENSOR if c["mode"] == "tensor" else None)
        sampled.append(got)
        for p, (D, g) in enumerate(zip(t.D, t.gamma)):
            a = _System(c, t, D, g, tensor, _velocity(t) if c["mode"] == "flow" else None, device)
            new.append(a.solve(torch.from_numpy(u[p]).to(device), c["mode"] != "flow").reshape(-1).cpu().numpy())
    out = {"fields": np.concatenate(new)}
    if c["mode"] != "vectors":
        out["sampled"], out["counts"] = np.concatenate(sampled), None
    if c["mode"] == "channels":
        out["channels"] = None
    return out
