"""Which solver a step takes, on both sides of every limit of the fast solver.
The Krylov solvers finish their sums by launches of their own (KERNEL_FINISH),
the fast solver has none.  And the multigrid solvers' own tests, which batches
with default options no longer reach, with a cycle set (a coarsest level of at
most 255 nodes for 256)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, H = 0.1, 0.125


def _fast(eqf, fb, n):
    """One step from random fields: whether it was the fast solver's."""
    fb.profile(eqf.KERNEL_FINISH)
    for p in range(n):
        fb.upload(p, np.random.default_rng(p).random(fb.num_nodes(p)))
    assert fb.step().nconverged == n
    return fb.profile_read(eqf.KERNEL_FINISH)[0] == 0


@pytest.mark.parametrize("kind", ["GMG_CG", "MIXED_GMG_CG", "IR_GMG_CG"])
@pytest.mark.parametrize("nx,ny,D,options,fast", [
    (90, 44, 60.0, {}, True), (90, 44, 1.01 * H * H / DT, {}, True), (90, 44, 0.99 * H * H / DT, {}, False),
    (16, 4095, 40.0, {}, True), (16, 4096, 40.0, {}, False), (8192, 3, 40.0, {}, None), (8193, 3, 40.0, {}, False),
    (90, 44, 60.0, {"mg_pre": 3}, False), (90, 44, 60.0, {"mg_level_fused": 0}, False),
    (90, 44, 60.0, {"streams": 1, "check_every": 2, "use_graphs": 0}, True)])
def test_grids_and_options(eqf, kind, nx, ny, D, options, fast):
    """(8192 columns fit a block in single precision only: 16384 points.)"""
    d = eqf.field_desc(nx, ny, nx * H, ny * H, DT, D, 0.0, 0.0, {eqf.TOP: (eqf.DIRICHLET, 0.0, 0.0, 0.0)})
    with eqf.FieldBatch([d], solver=eqf.solver_desc(getattr(eqf, kind), **options)) as fb:
        assert _fast(eqf, fb, 1) == (kind != "GMG_CG" if fast is None else fast)


@pytest.mark.parametrize("kind,contrast,s,rate,limit,fast", [
    ("GMG_CG", 8.9, 0, 0, 64, True), ("GMG_CG", 9.1, 0, 0, 64, False), ("GMG_CG", 4.0, 0, 0, 63, False),
    ("IR_GMG_CG", 4.0, 0, 0, 64, False), ("MIXED_GMG_BICGSTAB", 0, 1.32, 0, 64, True),
    ("MIXED_GMG_BICGSTAB", 0, 1.34, 0, 64, False), ("GMG_BICGSTAB", 0, -1.32, 0, 64, True),
    ("MIXED_GMG_CG", 0, 0, 1.99, 64, True), ("MIXED_GMG_CG", 0, 0, 2.01, 64, False), ("IR_GMG_CG", 0, 0, 1.0, 64, False),
    ("GMG_CG", 4.0, 0, 0.5, 64, True), ("MIXED_GMG_BICGSTAB", 0, 0.3, 0.3, 64, True)])
def test_varying_coefficients(eqf, oracle, kind, contrast, s, rate, limit, fast):
    """Contrast, flow s and Robin part at their limits; a tensor and a flow
    with Robin walls on the left and right.  dt D = 2048 h^2 leaves the mass
    couplings 1e-4 of room at the limits.  Either way the step is the oracle's."""
    nx, ny, D = 64, 33, 2048 * H * H / DT
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    if rate:
        r = rate * np.sqrt(DT * D) * np.tanh(0.5 * nx * H / np.sqrt(DT * D)) / DT
        walls[oracle.LEFT] = walls[oracle.RIGHT] = (oracle.ROBIN, 0.0, r, 0.1)
    args = (nx, ny, nx * H, ny * H, DT, D, 0.0, 0.0)
    p = oracle.problem(*args, walls=walls)
    t = {}
    with eqf.FieldBatch([eqf.field_desc(*args, walls)], solver=eqf.solver_desc(getattr(eqf, kind), max_iter=limit)) as fb:
        n = fb.num_nodes(0)
        if contrast:
            v = np.random.default_rng(1).uniform(contrast ** -0.5, contrast ** 0.5, (2, n))
            v[:, 0] = contrast ** -0.5, contrast ** 0.5
            t = {"D11": v[0], "D22": v[1], "D12": 0 * v[0]}
            fb.set_tensor(0, *t.values())
        if s:
            vel = np.full(ny + 1, 2 * s * np.sqrt(D / DT))
            fb.set_velocity(0, vel)
            p.set_velocity(vel)
        assert _fast(eqf, fb, 1) == fast
        ref, _ = oracle.step(p, np.random.default_rng(0).random(n), "lu", **t)
        assert np.linalg.norm(fb.download(0) - ref) <= 1e-9 * np.linalg.norm(ref)


class _WithACycle:
    """The binding, its solvers with a cycle of their own."""

    def __init__(self, eqf):
        self._eqf = eqf

    def __getattr__(self, name):
        return getattr(self._eqf, name)

    def solver_desc(self, kind, **options):
        return self._eqf.solver_desc(kind, mg_coarse_max_nodes=255, **options)


@pytest.mark.parametrize("solver", ["gmg", "mixed"])
@pytest.mark.parametrize("traps,streams", [(1, 2), (3, 3)])
def test_problem_groups_of_the_cycles(eqf, oracle, solver, traps, streams):
    import test_gpu_parity
    test_gpu_parity.test_two_problem_groups_match_one(_WithACycle(eqf), oracle, solver, traps, streams)


def test_autotune_reaches_the_fast_solver(eqf):
    """A batch created with another cycle has no plans; one that autotune sets to
    the default cycle takes the fast solver like any other."""
    nx, ny = 300, 150
    d = eqf.field_desc(nx, ny, nx * H, ny * H, DT, 60.0, 0.0, 0.0, {eqf.TOP: (eqf.DIRICHLET, 0.0, 0.0, 0.0)})
    with eqf.FieldBatch([d], solver=eqf.solver_desc(eqf.MIXED_GMG_CG, mg_pre=3, mg_post=3)) as fb:
        assert not _fast(eqf, fb, 1)
        chosen = fb.autotune(2)
        default = eqf.solver_desc(eqf.MIXED_GMG_CG)
        same = all(getattr(chosen, k) == getattr(default, k) for k, _ in default._fields_)
        assert _fast(eqf, fb, 1) == same
