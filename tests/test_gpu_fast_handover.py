"""Where the fast solver does not reach the tolerance the multigrid solver takes
the step over, from fields that the fast solver left as they were."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, H = 0.1, 0.125


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("solver", ["GMG_CG", "MIXED_GMG_CG"])
@pytest.mark.parametrize("spare", [0, 1])
def test_iteration_limits_that_the_cycles_meet(eqf, oracle, solver, spare):
    """dt D near the square of the spacing, where an application gains least:
    an iteration limit that the V-cycle CG needs no more than (its own count,
    from a batch with a cycle set) is enough."""
    nx, ny = 90, 44
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    args = (nx, ny, nx * H, ny * H, DT, 1.1 * H * H / DT, 0.01, 0.0)
    u = np.random.default_rng(2).random((nx + 1) * (ny + 1))
    ref, _ = oracle.step(oracle.problem(*args, walls=walls), u, "lu")
    kind = getattr(eqf, solver)
    with eqf.FieldBatch([eqf.field_desc(*args, walls)], solver=eqf.solver_desc(kind, mg_coarse_max_nodes=255)) as fb:
        fb.upload(0, u)
        need = fb.step().iterations_max
    with eqf.FieldBatch([eqf.field_desc(*args, walls)], solver=eqf.solver_desc(kind, max_iter=need + spare)) as fb:
        fb.upload(0, u)
        assert fb.step().nconverged == 1, need
        assert _rel(fb.download(0), ref) <= 1e-9


@pytest.mark.parametrize("solver", ["GMG_CG", "MIXED_GMG_CG"])
def test_a_tensor_set_over_the_cells_tensor(eqf, oracle, solver):
    """A tensor field set on a problem whose cells drive its tensor, then rods
    that write it again: the operator's eigenvalues are the cells', not the set
    field's.  Each step, from a kept solution and after a step that went wrong
    or right, is the oracle's, by no more applications than with the cells'
    tensor alone (a diverging solve takes 64, then cycles)."""
    import torch
    nx, ny, npm = 96, 48, 8.0
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    args = (nx, ny, nx / npm, ny / npm, DT, 60.0, 0.01, 0.0)
    rng = np.random.default_rng(3)
    n, nc = (nx + 1) * (ny + 1), 60
    cells = np.column_stack([rng.uniform(0, nx / npm, nc), rng.uniform(0, ny / npm, nc), rng.uniform(0, 3, nc),
                             rng.uniform(2, 4, nc), np.ones(nc)])
    u = rng.random(n)
    cells_d = torch.from_numpy(cells).cuda()
    q_d = torch.from_numpy(rng.random((nc, 1)) * 0.1).cuda()
    samp = torch.zeros((nc, 1), dtype=torch.float64, device="cuda")
    cnt = torch.zeros(nc, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    p = oracle.problem(*args, walls=walls)
    with eqf.FieldBatch([eqf.field_desc(*args, walls)], solver=eqf.solver_desc(getattr(eqf, solver))) as fb:
        fb.profile(eqf.KERNEL_FINISH)
        fb.upload(0, u)
        its = []
        fb.cell_tensor(0, 7.0, 1.0)
        for step in range(4):
            if step == 2:
                fb.set_tensor(0, np.ones(n), np.ones(n), np.zeros(n))
            fb.couple_dev(0, cells_d.data_ptr(), nc, npm, q_d.data_ptr(), samp.data_ptr(), cnt.data_ptr(),
                          eqf.SAMPLE | eqf.DEPOSIT | eqf.TENSOR)
            before, t = fb.download(0), fb.tensor_values(0)
            st = fb.step()
            assert st.nconverged == 1, step
            its.append(st.iterations_max)
            # the fast solver's steps, and it alone: the Krylov solvers finish their sums by launches of their own
            assert fb.profile_read(eqf.KERNEL_FINISH)[0] == 0 and its[step] <= max(its[:2]), its
            ref, _ = oracle.step(p, before, "lu", D11=t[0], D22=t[1], D12=t[2])
            assert _rel(fb.download(0), ref) <= 1e-9, step


def test_a_refused_tensor_leaves_the_other_problems(eqf, oracle):
    """A tensor that is refused (not positive definite, found out level by
    level) beside a problem with a velocity, which the fast solver would take:
    that problem's steps stay the oracle's, before and after the tensor is
    taken off again."""
    nx, ny = 64, 33
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    args = (nx, ny, nx * H, ny * H, DT, 60.0, 0.01, 0.0)
    rng = np.random.default_rng(4)
    u, vel, one = rng.random((nx + 1) * (ny + 1)), 10.0 * rng.random(ny + 1), np.ones((nx + 1) * (ny + 1))
    p = oracle.problem(*args, walls=walls)
    p.set_velocity(vel)
    with eqf.FieldBatch([eqf.field_desc(*args, walls)] * 2,
                        solver=eqf.solver_desc(eqf.GMG_BICGSTAB, max_iter=100)) as fb:
        fb.set_velocity(0, vel)
        for step in range(3):
            if step == 1:
                with pytest.raises(eqf.EqError) as e:
                    fb.set_tensor(1, -one, -one, 0.0 * one)
                assert e.value.code == 1
            if step == 2:
                fb.set_tensor(1)
            fb.upload(0, u)
            fb.upload(1, u)
            st = fb.step(check=False)
            assert st.nconverged == (1 if step == 1 else 2), step
            ref, _ = oracle.step(p, u, "lu")
            assert _rel(fb.download(0), ref) <= 1e-9, step


@pytest.mark.parametrize("kind,nx,ny,walls,flow,fast", [
    ("GMG_BICGSTAB", 404, 154, "top", True, True), ("GMG_BICGSTAB", 1237, 611, "top", True, False),
    ("MIXED_GMG_BICGSTAB", 901, 449, "top", True, True), ("MIXED_GMG_BICGSTAB", 2999, 1000, "top", True, False),
    ("GMG_BICGSTAB", 2999, 1000, "top", False, True), ("GMG_CG", 404, 154, "sides", False, True),
    ("GMG_CG", 2999, 1800, "sides", False, False), ("MIXED_GMG_CG", 2999, 1800, "top", False, True)])
def test_the_faster_solver_is_taken(eqf, oracle, kind, nx, ny, walls, flow, fast):
    """Flow and Robin walls across x go by the measured times of both solvers;
    without either every size is the fast solver's."""
    w = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    if walls == "sides":
        w[oracle.LEFT] = w[oracle.RIGHT] = (oracle.ROBIN, 0.0, 1.5, 0.2)
    descs = [eqf.field_desc(nx, ny, nx * 0.1, ny * 0.1, DT, D, 0.01, 0.0, w) for D in (400.0, 100.0)]
    y = np.linspace(0, 1, ny + 1)
    with eqf.FieldBatch(descs, nspecies=2, solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        fb.profile(eqf.KERNEL_FINISH)
        for p in range(2):
            if flow:
                fb.set_velocity(p, 200.0 * y * (1 - y))
            fb.upload(p, np.random.default_rng(p).random((nx + 1) * (ny + 1)))
        assert fb.step().nconverged == 2
        assert (fb.profile_read(eqf.KERNEL_FINISH)[0] == 0) == fast


def test_a_give_up_is_remembered(eqf, oracle):
    """A tolerance below rounding: the fast solver tries again after 1, 3, 7, ...
    steps of the cycles.  A try shows in the launches of the updates: 32 more."""
    nx, ny = 70, 41
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    d = eqf.field_desc(nx, ny, nx * H, ny * H, DT, 60.0, 0.01, 0.0, walls)
    u = np.random.default_rng(1).random((nx + 1) * (ny + 1))
    counts = []
    with eqf.FieldBatch([d], solver=eqf.solver_desc(eqf.GMG_CG, rtol=1e-18, max_iter=40)) as fb:
        fb.profile(eqf.KERNEL_CG_UPDATE)
        fb.upload(0, u)
        for step in range(12):
            before = fb.profile_read(eqf.KERNEL_CG_UPDATE)[0]
            fb.step(check=False)
            counts.append(fb.profile_read(eqf.KERNEL_CG_UPDATE)[0] - before)
    # (step 0 tries too, and has fewer cycles)
    assert [k for k in range(1, 12) if counts[k] >= counts[1] + 32] == [2, 6], counts


def test_refinement_after_a_hand_over(eqf, oracle):
    """IR_GMG_CG at a tolerance below rounding: its own refinement runs out too,
    and reports its inner iterations, of the problem that needed them."""
    nx, ny = 70, 41
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    args = (nx, ny, nx * H, ny * H, DT, 60.0, 0.01, 0.0)
    u = np.random.default_rng(1).random((nx + 1) * (ny + 1))
    with eqf.FieldBatch([eqf.field_desc(*args, walls)] * 2, nspecies=2,
                        solver=eqf.solver_desc(eqf.IR_GMG_CG, rtol=1e-18)) as fb:
        fb.upload(0, np.zeros_like(u))
        fb.upload(1, u)
        st = fb.step(check=False)
        its = fb.problem_stats()[0]
        assert st.nconverged == 1 and its[0] == 0 and st.iterations_max == its[1] > 20, its
        assert not fb.download(0).any()
        ref, _ = oracle.step(oracle.problem(*args, walls=walls), u, "lu")
        assert _rel(fb.download(1), ref) <= 1e-9


@pytest.mark.parametrize("kind", ["GMG_CG", "MIXED_GMG_CG", "IR_GMG_CG"])
@pytest.mark.parametrize("spoil", ["infinity", "nan", "large"])
def test_fields_without_a_finite_norm(eqf, oracle, kind, spoil):
    """An infinity or a NaN in a fresh field, and values whose squares overflow,
    end as they do with the cycles: the same error, or the same field."""
    nx, ny = 70, 41
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    d = eqf.field_desc(nx, ny, nx * H, ny * H, DT, 60.0, 0.01, 0.0, walls)
    u = np.random.default_rng(6).random((nx + 1) * (ny + 1))
    u[-(nx + 1):] = 0.0
    if spoil == "large":
        u = np.ldexp(u, 600)
    else:
        u[500] = {"infinity": np.inf, "nan": np.nan}[spoil]
    ends = []
    for options in ({}, {"mg_coarse_max_nodes": 255}):
        with eqf.FieldBatch([d], solver=eqf.solver_desc(getattr(eqf, kind), max_iter=70, **options)) as fb:
            fb.upload(0, u)
            try:
                fb.step()
                ends.append(fb.download(0))
            except eqf.EqError as e:
                ends.append(np.array([float(e.code)]))
    assert np.array_equal(*ends), [e[:3] for e in ends]
