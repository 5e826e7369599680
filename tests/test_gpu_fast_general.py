"""The fast solver where coefficients vary (Chebyshev iteration on the constant
operator): tensor fields and velocities on both sides of the bounds that choose
it (contrast 9, s = 4/3), either flow direction, problems with and without in
one batch, changes between steps, stopping at the iteration limit's rule.  Each
step is within 1e-9 relative L2 of the oracle's direct solve: the bar of every
solve at rtol 1e-10 on these grids."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, H = 0.1, 0.125
SHAPES = [(37, 20), (64, 33), (105, 16), (3, 5), (256, 9)]


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def _walls(o, kind):
    d, r = (o.DIRICHLET, 0.25, 0.0, 0.0), (o.ROBIN, 0.0, 1.5, 0.2)
    return {"top": {o.TOP: d}, "sides": {o.LEFT: d, o.RIGHT: d, o.BOTTOM: r}, "mixed": {o.RIGHT: d, o.TOP: r}}[kind]


def _tensor(rng, n, contrast):
    """Eigenvalues between 1/sqrt(contrast) and sqrt(contrast), any direction."""
    c = np.sqrt(contrast)
    a, b, t = rng.uniform(1 / c, c, n), rng.uniform(1 / c, c, n), rng.uniform(0, np.pi, n)
    a[0], b[0] = 1 / c, c
    cs, sn = np.cos(t), np.sin(t)
    return a * cs * cs + b * sn * sn, a * sn * sn + b * cs * cs, (a - b) * sn * cs


@pytest.mark.parametrize("kind", ["GMG_CG", "MIXED_GMG_CG"])
@pytest.mark.parametrize("walls", ["top", "sides", "mixed"])
@pytest.mark.parametrize("contrast", [2.0, 8.9, 9.5])
def test_tensor_fields(eqf, oracle, kind, walls, contrast):
    rng = np.random.default_rng(int(contrast * 10))
    w = _walls(oracle, walls)
    descs, args_of, u = [], [], []
    tens = [None] * len(SHAPES)
    for k, (nx, ny) in enumerate(SHAPES):
        args = (nx, ny, nx * H, ny * H, DT, 60.0 + 20 * k, 0.01, 0.05)
        descs.append(eqf.field_desc(*args, w))
        args_of.append(args)
        u.append(rng.random((nx + 1) * (ny + 1)))
    with eqf.FieldBatch(descs, solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k in range(len(descs)):
            fb.upload(k, u[k])
        for step in range(4):
            # every problem but the second; then constant again; then one alone
            for k in range(len(descs)):
                if step == 1:
                    continue
                tens[k] = _tensor(rng, u[k].size, contrast) if (step == 0 and k != 1) or (step == 3 and k == 2) else None
                fb.set_tensor(k, *(tens[k] or ()))
            assert fb.step().nconverged == len(descs)
            for k, a in enumerate(args_of):
                t = dict(zip(("D11", "D22", "D12"), tens[k] or ()))
                u[k], _ = oracle.step(oracle.problem(*a, walls=w), u[k], "lu", **t)
                assert _rel(fb.download(k), u[k]) <= 1e-9, (step, k)


@pytest.mark.parametrize("kind", ["GMG_BICGSTAB", "MIXED_GMG_BICGSTAB"])
@pytest.mark.parametrize("walls", ["top", "sides", "mixed"])
@pytest.mark.parametrize("s", [0.1, -0.8, 1.3, 1.4])
def test_velocities(eqf, oracle, kind, walls, s):
    rng = np.random.default_rng(int(abs(s) * 10))
    w = _walls(oracle, walls)
    descs, probs, u, vel = [], [], [], []
    for k, (nx, ny) in enumerate(SHAPES):
        D, gamma = 60.0 + 20 * k, 0.5
        args = (nx, ny, nx * H, ny * H, DT, D, gamma, 0.05)
        descs.append(eqf.field_desc(*args, w))
        probs.append(oracle.problem(*args, walls=w))
        u.append(rng.random((nx + 1) * (ny + 1)))
        y = np.arange(ny + 1) / ny
        vel.append(2.0 * s * np.sqrt((1 + DT * gamma) * D / DT) * (1.0 - (2 * y - 1) ** 2 / 2))
    with eqf.FieldBatch(descs, solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k in range(len(descs)):
            fb.upload(k, u[k])
        for step in range(3):
            for k, p in enumerate(probs):
                v = vel[k] if (step == 0 and k != 1) or (step == 2 and k == 2) else None
                fb.set_velocity(k, v)
                p.set_velocity(v)
            assert fb.step().nconverged == len(descs)
            for k, p in enumerate(probs):
                u[k], _ = oracle.step(p, u[k], "lu")
                assert _rel(fb.download(k), u[k]) <= 1e-9, (step, k)


def test_advection_still_needs_a_bicgstab_solver(eqf):
    with eqf.FieldBatch([eqf.field_desc(40, 20, 4.0, 2.0, DT, 100.0)], solver=eqf.solver_desc(eqf.GMG_CG)) as fb:
        fb.set_velocity(0, np.ones(21))
        with pytest.raises(eqf.EqError) as e:
            fb.step()
        assert e.value.code == 1


@pytest.mark.parametrize("kind", ["GMG_CG", "MIXED_GMG_CG", "MIXED_GMG_BICGSTAB"])
@pytest.mark.parametrize("left,right", [(1.5, 1.5), (0.0, 1.5), (None, 30.0), (50.0, None), (60.0, 400.0)])
@pytest.mark.parametrize("fd", [False, True])
def test_robin_walls_across_x(eqf, oracle, kind, left, right, fd):
    """Rates from none to past the bound (twice the closed operator), one or
    both walls, the other held; a step of every kind with them."""
    w = {oracle.TOP: (oracle.DIRICHLET, 0.25, 0.0, 0.0)}
    for wall, r in ((oracle.LEFT, left), (oracle.RIGHT, right)):
        w[wall] = (oracle.DIRICHLET, 0.5, 0.0, 0.0) if r is None else (oracle.ROBIN, 0.0, r, 0.2)
    rng = np.random.default_rng(11)
    descs, probs, u = [], [], []
    for k, (nx, ny) in enumerate(SHAPES):
        # (the finite-difference oracle has no reaction and no source)
        args = (nx, ny, nx * H, ny * H, DT, 60.0 + 20 * k) + ((0.0, 0.0) if fd else (0.01, 0.05))
        descs.append(eqf.field_desc(*args, w, scheme=eqf.SCHEME_FD if fd else eqf.SCHEME_P1))
        probs.append(oracle.problem(*args, walls=w))
        u.append(rng.random((nx + 1) * (ny + 1)))
    with eqf.FieldBatch(descs, solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k in range(len(descs)):
            fb.upload(k, u[k])
        for step in range(2):
            assert fb.step().nconverged == len(descs)
            for k, p in enumerate(probs):
                u[k] = oracle.fd_step(p, u[k]) if fd else oracle.step(p, u[k], "lu")[0]
                assert _rel(fb.download(k), u[k]) <= 1e-9, (step, k)
