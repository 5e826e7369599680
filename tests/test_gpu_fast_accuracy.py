"""How far the fast solver's steps are from a 64-bit direct solve (refined on
residuals in extended precision).  The V-cycle CG and BiCGStab at rtol 1e-10 leave
4e-14 to 1e-13 of fields like these (smooth, with deposits); no step may leave
more than 1e-13."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 0.1


def _operator(nx, ny, w, h, D, gamma, vel=None, robin=0.0):
    """x -> (mass M x, operator A x) of the P1 "right"-diagonal mesh with closed walls, or Robin walls (s = 0) of that
    rate on the left and right, in extended precision.  The
    stiffness takes differences: entries rounded to 64 bits alone are worth 1e-12 of the solution at dt D = 6000 h^2."""
    hx, hy = np.longdouble(w) / nx, np.longdouble(h) / ny
    area = hx * hy / 2
    v = None if vel is None else np.repeat(vel.astype(np.longdouble)[:, None], nx + 1, 1)
    tri = ((((0, 0), (0, 1), (1, 1)), ((-1 / hx, 0), (1 / hx, -1 / hy), (0, 1 / hy))),
           (((0, 0), (1, 0), (1, 1)), ((0, -1 / hy), (-1 / hx, 1 / hy), (1 / hx, 0))))

    def both(x):
        x = x.reshape(ny + 1, nx + 1)
        at = lambda a, p: a[p[0]:ny + p[0], p[1]:nx + p[1]]  # noqa: E731
        m, k = np.zeros_like(x), np.zeros_like(x)
        for verts, grads in tri:
            for pa, ga in zip(verts, grads):
                for pb, gb in zip(verts, grads):
                    at(m, pa)[...] += area / (6 if pa == pb else 12) * at(x, pb)
                    if pa == pb:
                        continue
                    c = np.longdouble(D) * area * (ga[0] * gb[0] + ga[1] * gb[1])
                    if v is not None:
                        c = c + gb[0] * area / 12 * (sum(at(v, p) for p in verts) + at(v, pa))
                    at(k, pa)[...] += c * (at(x, pb) - at(x, pa))
        for e in (0, -1):
            at = x[:, e]
            k[:-1, e] += robin * hy * (at[:-1] / 3 + at[1:] / 6)
            k[1:, e] += robin * hy * (at[1:] / 3 + at[:-1] / 6)
        return m.reshape(-1), ((1 + np.longdouble(DT) * gamma) * m + np.longdouble(DT) * k).reshape(-1)
    return both


def _exact(o, p, a, u, vel=None, robin=0.0):
    """The step's solution with the top wall held at 0: the oracle's matrix factored, refined on extended residuals."""
    import scipy.sparse.linalg as sla
    rp, c, v = o.assemble(p)
    v, _ = o.apply_dirichlet(p, rp, c, v, o.assemble_rhs(p, u))
    lu = sla.splu(o.to_scipy(rp, c, v, u.size).tocsc())
    both = _operator(*a[:4], a[5], a[6], vel, robin)
    b = both(u.astype(np.longdouble))[0]
    x = np.zeros(u.size, np.longdouble)
    for _ in range(4):
        r = b - both(x)[1]
        r[-(a[0] + 1):] = 0
        x = x + lu.solve(r.astype(np.float64))
    return x


def _field(rng, nx, ny):
    x, y = np.linspace(0, 1, nx + 1)[None, :], np.linspace(0, 1, ny + 1)[:, None]
    u = 0.02 * (1 + 0.3 * np.cos(np.pi * x) * np.cos(2 * np.pi * y)) * np.sin(0.5 * np.pi * (1 - y))
    for _ in range(nx * ny // 400):
        i, j = rng.integers(1, ny - 9), rng.integers(1, nx - 9)
        u[i:i + 8, j:j + 8] += rng.uniform(0.5, 1.5) * DT / 64
    u[-1] = 0.0
    return u.reshape(-1)


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("kind", ["MIXED_GMG_CG", "GMG_CG"])
def test_uneven_traps(eqf, oracle, kind):
    rng = np.random.default_rng(21)
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    args = []
    for _ in range(8):
        nx, ny = int(rng.integers(200, 420)), int(rng.integers(100, 200))
        args += [(nx, ny, nx / 10, ny / 10, DT, rng.uniform(*r), 0.01, 0.0) for r in ((200, 600), (50, 150))]
    u = [_field(rng, a[0], a[1]) for a in args]
    with eqf.FieldBatch([eqf.field_desc(*a, walls) for a in args], nspecies=2,
                        solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k, x in enumerate(u):
            fb.upload(k, x)
        fb.step()
        err = [_rel(fb.download(k), _exact(oracle, oracle.problem(*a, walls=walls, grid_walls=True), a, u[k])) for k, a in enumerate(args)]
    assert max(err) <= 1e-13, err


@pytest.mark.parametrize("kind", ["MIXED_GMG_BICGSTAB", "GMG_BICGSTAB"])
def test_velocities(eqf, oracle, kind):
    """A channel's profile at s = 0.8 and 0.4 for the two species; the first
    step, and one from a kept solution."""
    rng = np.random.default_rng(22)
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    nx, ny = 301, 149
    args = [(nx, ny, nx / 20, ny / 20, DT, D, 0.01, 0.0) for D in (400.0, 100.0)]
    y = np.linspace(0, 1, ny + 1)
    vel = 200.0 * y * (1 - y)
    u = [_field(rng, nx, ny) for _ in args]
    probs = [oracle.problem(*a, walls=walls, grid_walls=True) for a in args]
    with eqf.FieldBatch([eqf.field_desc(*a, walls) for a in args], nspecies=2,
                        solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k, p in enumerate(probs):
            fb.set_velocity(k, vel)
            p.set_velocity(vel)
            fb.upload(k, u[k])
        for step in range(2):
            fb.step()
            for k, a in enumerate(args):
                ref = _exact(oracle, probs[k], a, u[k], vel)
                u[k] = fb.download(k)
                assert _rel(u[k], ref) <= 1e-13, (step, k)


@pytest.mark.parametrize("kind", ["MIXED_GMG_CG", "GMG_CG"])
def test_robin_walls(eqf, oracle, kind):
    rng = np.random.default_rng(23)
    rate = 1.5
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0), oracle.LEFT: (oracle.ROBIN, 0.0, rate, 0.0),
             oracle.RIGHT: (oracle.ROBIN, 0.0, rate, 0.0)}
    nx, ny = 227, 128
    args = [(nx, ny, nx / 10, ny / 10, DT, D, 0.01, 0.0) for D in (400.0, 100.0, 250.0)]
    u = [_field(rng, nx, ny) for _ in args]
    with eqf.FieldBatch([eqf.field_desc(*a, walls) for a in args], nspecies=3,
                        solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k, x in enumerate(u):
            fb.upload(k, x)
        for step in range(2):
            fb.step()
            for k, a in enumerate(args):
                ref = _exact(oracle, oracle.problem(*a, walls=walls, grid_walls=True), a, u[k], robin=rate)
                u[k] = fb.download(k)
                assert _rel(u[k], ref) <= 1e-13, (step, k)
