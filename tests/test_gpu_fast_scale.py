"""The single-precision kinds of the fast solver at any magnitude of the field:
a problem without sources is linear and every scale here is a power of two, so
the solution is the unscaled one times that scale, bit for bit, in as many
applications (FP64 sums of squares stay above 2^-1022).  Scales change both ways
within one batch, with and without a kept solution; constant coefficients, a
tensor field and a velocity.  Then a field that only decays, over 2000 steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, H = 0.1, 0.125
SHAPES = [(37, 40), (64, 33), (105, 16)]


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("kind,field", [("MIXED_GMG_CG", None), ("IR_GMG_CG", None), ("GMG_CG", None),
                                        ("MIXED_GMG_CG", "tensor"), ("MIXED_GMG_BICGSTAB", "velocity"),
                                        ("MIXED_GMG_BICGSTAB", None)])
def test_scaled_fields(eqf, oracle, kind, field):
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    rng = np.random.default_rng(7)
    args = [(nx, ny, nx * H, ny * H, DT, 60.0 + 40 * k, 0.01, 0.0) for k, (nx, ny) in enumerate(SHAPES)]
    u = [rng.random((a[0] + 1) * (a[1] + 1)) for a in args]
    extra = [{} for _ in args]
    probs = [oracle.problem(*a, walls=walls) for a in args]
    with eqf.FieldBatch([eqf.field_desc(*a, walls) for a in args], solver=eqf.solver_desc(getattr(eqf, kind))) as fb:
        for k, a in enumerate(args):
            if field == "tensor":
                d = rng.uniform(0.6, 1.6, (2, u[k].size))
                extra[k] = {"D11": d[0], "D22": d[1], "D12": 0.0 * d[0]}
                fb.set_tensor(k, *extra[k].values())
            if field == "velocity":
                v = 20.0 * rng.random(a[1] + 1)
                fb.set_velocity(k, v)
                probs[k].set_velocity(v)
        base = None
        for e in (0, -100, -101, 100, -200, -400, 300, -60, 0):
            got = []
            for k, x in enumerate(u):
                fb.upload(k, np.ldexp(x, e))
            for step in range(2):
                assert fb.step().nconverged == len(args), (e, step)
                got.append(([np.ldexp(fb.download(k), -e) for k in range(len(args))], list(fb.problem_stats()[0])))
            if base is None:
                base = got
                for k, p in enumerate(probs):
                    ref, _ = oracle.step(p, u[k], "lu", **extra[k])
                    assert _rel(got[0][0][k], ref) <= 1e-9, k
            for step in range(2):
                assert got[step][1] == base[step][1], (e, step)
                for k in range(len(args)):
                    assert np.array_equal(got[step][0][k], base[step][0][k]), (e, step, k)


@pytest.mark.parametrize("kind", ["MIXED_GMG_CG", "IR_GMG_CG", "GMG_CG", "MIXED_GMG_BICGSTAB"])
def test_decaying_field(eqf, oracle, kind):
    """A field without sources falls to 0.8 of itself a step, below every square
    that FP64 holds: no step errors.  After 300 steps (1e-29) the field is
    within 300 steps of 1e-10 of the FP64 kind's, with a factor of three."""
    nx, ny = 20, 160
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0.0, 0.0)}
    d = eqf.field_desc(nx, ny, nx * H, ny * H, DT, 400.0, 0.01, 0.0, walls)
    u = np.random.default_rng(9).random((nx + 1) * (ny + 1))
    at = {}
    for name in {kind, "GMG_CG"}:
        with eqf.FieldBatch([d], solver=eqf.solver_desc(getattr(eqf, name))) as fb:
            fb.upload(0, u)
            for step in range(2000 if name == kind else 300):
                st = fb.step()
                assert st.nconverged == 1, step
                if step == 299:
                    at[name] = fb.download(0)
            if name == kind:
                assert np.isfinite(fb.download(0)).all()
    assert 1e-33 < np.abs(at["GMG_CG"]).max() < 1e-25
    assert _rel(at[kind], at["GMG_CG"]) <= 1e-7
