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
