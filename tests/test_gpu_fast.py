"""The fast direct solver of constant-coefficient batches (transform along x,
one tridiagonal solve along y per mode) against the oracle's direct solve, at
the sizes where its kernels change shape: transform lengths with and without
prime factors above 7 (Stockham or chirp), the block sizes' edges, the line
solve's chunk lengths, every pair of x walls, Robin y walls, both schemes.
Steps are within 1e-9 relative L2 of the direct solve: the bar of every solve
at rtol 1e-10 on these grids (test_gpu_parity)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOLVERS = ["gmg", "mixed"]
H = 0.125  # every node coordinate exact


def _kind(eqf, name):
    return {"gmg": eqf.GMG_CG, "mixed": eqf.MIXED_GMG_CG}[name]


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def _walls(o, left, right, bottom="N", top="D"):
    kinds = {"N": (o.NEUMANN, 0.0, 0.0, 0.0), "D": (o.DIRICHLET, 0.25, 0.0, 0.0), "R": (o.ROBIN, 0.0, 1.5, 0.2)}
    return {o.LEFT: kinds[left], o.RIGHT: kinds[right], o.BOTTOM: kinds[bottom], o.TOP: kinds[top]}


@pytest.mark.parametrize("solver", SOLVERS)
@pytest.mark.parametrize("left,right,bottom,top", [("N", "N", "N", "D"), ("D", "D", "R", "N"), ("N", "D", "D", "R"),
                                                   ("D", "N", "N", "N"), ("N", "N", "R", "R")])
def test_walls_and_lengths(eqf, oracle, solver, left, right, bottom, top):
    """One batch per set of walls: transform lengths 2 nx of factors 2, 3, 5, 7
    and with primes (chirp), nx = 1, odd and even row counts; three steps, the
    second from the kept solution, the third after new wall values."""
    shapes = [(1, 3), (2, 1), (37, 20), (64, 33), (94, 15), (105, 16), (256, 17), (257, 9)]
    walls = _walls(oracle, left, right, bottom, top)
    descs, probs, u = [], [], []
    rng = np.random.default_rng(3)
    for nx, ny in shapes:
        for D in (300.0, 2.0):
            descs.append(eqf.field_desc(nx, ny, nx * H, ny * H, 0.1, D, 0.02, 0.1, walls))
            probs.append(oracle.problem(nx, ny, nx * H, ny * H, 0.1, D, 0.02, 0.1, walls=walls))
            u.append(rng.random((nx + 1) * (ny + 1)))
    with eqf.FieldBatch(descs, nspecies=2, solver=eqf.solver_desc(_kind(eqf, solver))) as fb:
        for p, x in enumerate(u):
            fb.upload(p, x)
        for step in range(3):
            if step == 2 and top == "D":
                for p, (nx, ny) in enumerate(s for s in shapes for _ in range(2)):
                    g = np.linspace(0.0, 1.0, nx + 1)
                    fb.set_wall_values(p, oracle.TOP, g)
                    probs[p].set_wall_values(oracle.TOP, g)
            st = fb.step()
            assert st.nconverged == len(descs) and st.relres_max <= 1e-10
            for p in range(len(descs)):
                u[p], _ = oracle.step(probs[p], u[p], "lu")
                assert _rel(fb.download(p), u[p]) <= 1e-9, (step, p)


@pytest.mark.parametrize("solver", SOLVERS)
def test_finite_differences(eqf, oracle, solver):
    """The 5-point scheme is separable exactly: held, closed and Robin walls."""
    shapes = [(48, 31), (53, 40)]
    descs, probs, u = [], [], []
    rng = np.random.default_rng(5)
    for nx, ny in shapes:
        for left, right, bottom, top in (("N", "N", "R", "D"), ("D", "N", "N", "R"), ("D", "D", "D", "N")):
            walls = _walls(oracle, left, right, bottom, top)
            descs.append(eqf.field_desc(nx, ny, nx * H, ny * H, 0.1, 80.0, 0.0, 0.0, walls, scheme=eqf.SCHEME_FD))
            probs.append(oracle.problem(nx, ny, nx * H, ny * H, 0.1, 80.0, 0.0, 0.0, walls=walls))
            u.append(rng.random((nx + 1) * (ny + 1)))
    with eqf.FieldBatch(descs, nspecies=3, solver=eqf.solver_desc(_kind(eqf, solver))) as fb:
        for p, x in enumerate(u):
            fb.upload(p, x)
        for step in range(2):
            assert fb.step().nconverged == len(descs)
            for p in range(len(descs)):
                u[p] = oracle.fd_step(probs[p], u[p])
                assert _rel(fb.download(p), u[p]) <= 1e-9, (step, p)


@pytest.mark.parametrize("solver", SOLVERS)
@pytest.mark.parametrize("nx,ny", [(24, 1023), (24, 1024), (23, 2047), (24, 2048), (16, 4095), (16, 4096), (1024, 5),
                                   (2048, 4), (2400, 3), (2729, 3), (4096, 3), (4100, 3), (8191, 2), (9000, 2)])
def test_long_rows_and_columns(eqf, oracle, solver, nx, ny):
    """The edges of the blocks' ranges: row counts of 1024, 2048 and 4096 (the
    last the line solve takes) and one more, transform lengths at the thread
    counts' limits and past the LDS (the multigrid solver takes those)."""
    walls = _walls(oracle, "N", "N")
    d = eqf.field_desc(nx, ny, nx * H, ny * H, 0.1, 40.0, 0.01, 0.0, walls)
    p = oracle.problem(nx, ny, nx * H, ny * H, 0.1, 40.0, 0.01, 0.0, walls=walls)
    u = np.random.default_rng(nx + ny).random((nx + 1) * (ny + 1))
    rp, c, v = oracle.assemble(p)
    b = oracle.assemble_rhs(p, u)
    v, b = oracle.apply_dirichlet(p, rp, c, v, b)
    import scipy.sparse.linalg as sla
    ref = sla.spsolve(oracle.to_scipy(rp, c, v, u.size).tocsc(), b)
    with eqf.FieldBatch([d], solver=eqf.solver_desc(_kind(eqf, solver))) as fb:
        fb.upload(0, u)
        st = fb.step()
        assert st.nconverged == 1
        assert _rel(fb.download(0), ref) <= 1e-9


@pytest.mark.parametrize("solver", SOLVERS)
def test_takes_over_where_the_tolerance_is_out_of_reach(eqf, oracle, solver):
    """A tolerance below rounding: the problem that reaches it (a zero field)
    keeps its solution, the other goes on with the multigrid solver to
    max_iter, reports non-convergence and still holds the step's solution."""
    nx, ny = 70, 41
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    d = [eqf.field_desc(nx, ny, nx * H, ny * H, 0.1, 60.0, 0.01, 0.0, walls) for _ in range(2)]
    p = oracle.problem(nx, ny, nx * H, ny * H, 0.1, 60.0, 0.01, 0.0, walls=walls)
    u = np.random.default_rng(1).random((nx + 1) * (ny + 1))
    with eqf.FieldBatch(d, nspecies=2, solver=eqf.solver_desc(_kind(eqf, solver), rtol=1e-18, max_iter=60)) as fb:
        fb.upload(0, np.zeros_like(u))
        fb.upload(1, u)
        with pytest.raises(eqf.EqError) as e:
            fb.step()
        assert e.value.code == 4
        assert not fb.download(0).any()
        ref, _ = oracle.step(p, u, "lu")
        assert _rel(fb.download(1), ref) <= 1e-9
        assert list(fb.problem_stats()[0]) == [0, 60]


def test_small_time_steps_and_set_cycles_keep_multigrid(eqf, oracle):
    """dt D below the square of the spacing, and a caller's own cycle options,
    stay with the multigrid solver: the step is the same either way."""
    nx, ny = 90, 44
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    u = np.random.default_rng(2).random((nx + 1) * (ny + 1))
    for D, kw in ((0.1, {}), (60.0, {"mg_pre": 3, "mg_post": 3}), (60.0, {"mg_level_fused": 0}), (60.0, {})):
        d = eqf.field_desc(nx, ny, nx * H, ny * H, 0.1, D, 0.01, 0.0, walls)
        p = oracle.problem(nx, ny, nx * H, ny * H, 0.1, D, 0.01, 0.0, walls=walls)
        with eqf.FieldBatch([d], solver=eqf.solver_desc(eqf.MIXED_GMG_CG, **kw)) as fb:
            fb.upload(0, u)
            assert fb.step().nconverged == 1
            ref, _ = oracle.step(p, u, "lu")
            assert _rel(fb.download(0), ref) <= 1e-9, (D, kw)
