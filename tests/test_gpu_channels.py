"""The flow channels' block scans at the sizes where their rows change shape: one
element, one row a thread and its edges (512 threads), several rows a thread.
Channel values after each step against the oracle's update from the step's own
field, within 1e-11 relative L2: the substep's matrix has a condition number of
at most 1 + 4 k D / h^2 (1.2e4 here), which times the unit roundoff over nine
substeps is 1.2e-11 at the worst alignment."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [1, 2, 510, 511, 512, 1023, 1537])
def test_channel_sizes(eqf, oracle, nx):
    ny, h = 6, 0.1
    walls = {oracle.TOP: (oracle.DIRICHLET, 0.0, 0, 0), oracle.BOTTOM: (oracle.DIRICHLET, 0.0, 0, 0)}
    args = (nx, ny, nx * h, ny * h, 0.1, 300.0, 0.01, 0.0)
    p = oracle.problem(*args, walls=walls)
    chans = [(35.0, 60.0, 0.1, 42.0, 0.0, 2.5, 3), (0.0, 60.0, 0.0, 42.0, 0.2, 2.5, 1)]
    u = np.random.default_rng(nx).random((nx + 1) * (ny + 1))
    top, bot = np.zeros(nx + 1), np.zeros(nx + 1)
    with eqf.FieldBatch([eqf.field_desc(*args, walls)], solver=eqf.solver_desc(eqf.GMG_CG)) as fb:
        fb.set_channels(0, eqf.channel_desc(*chans[0]), eqf.channel_desc(*chans[1]))
        fb.upload(0, u)
        for step in range(3):
            fb.step()
            top, bot = oracle.channel_update(p, oracle.channel(*chans[0]), oracle.channel(*chans[1]), fb.download(0),
                                             top, bot)
            got = fb.channel_values(0)
            for a, b in zip(got, (top, bot)):
                assert np.linalg.norm(a - b) <= 1e-11 * np.linalg.norm(b), step
