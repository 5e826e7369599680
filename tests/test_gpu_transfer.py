"""Fields and host arrays through the pinned staging at its edges: fields below,
at and across the 131072-word buffers, several chunks in one direction, odd row
lengths, host and device round trips (bytes exact), an upload as a new state,
a coupling whose arrays outgrow the kept device buffer's first size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 6), (254, 513), (511, 255), (1022, 600), (65535, 3), (65536, 5)])
def test_round_trips(eqf, nx, ny):
    import torch
    n = (nx + 1) * (ny + 1)
    descs = [eqf.field_desc(nx, ny, nx * 0.1, ny * 0.1, 0.1, 100.0)] * 2
    rng = np.random.default_rng(nx)
    u = [rng.random(n), rng.random(n)]
    with eqf.FieldBatch(descs, nspecies=2, solver=eqf.solver_desc(eqf.GMG_CG)) as fb:
        for p in range(2):
            fb.upload(p, u[p])
        for p in range(2):
            assert np.array_equal(fb.download(p), u[p])
        d = torch.full((n + 2,), -7.0, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        fb.download_dev(0, d.data_ptr() + 8, n)
        fb.sync()
        got = d.cpu().numpy()
        assert np.array_equal(got[1:-1], u[0]) and got[0] == got[-1] == -7.0
        fb.upload_dev(1, d.data_ptr() + 8, n)
        fb.sync()
        assert np.array_equal(fb.download(1), u[0]) and np.array_equal(fb.download(0), u[0])


def test_host_coupling_sizes(eqf, oracle):
    nx, ny, npm = 200, 100, 10.0
    grid = oracle.grid(nx + 1, ny + 1, npm, 20.0, 10.0)
    rng = np.random.default_rng(8)
    u0 = rng.random((nx + 1) * (ny + 1))
    with eqf.FieldBatch([eqf.field_desc(nx, ny, 20.0, 10.0, 0.1, 100.0)], solver=eqf.solver_desc(eqf.GMG_CG)) as fb:
        for nc in (3, 5000, 1, 28001):
            c = np.column_stack([rng.uniform(0, 20, nc), rng.uniform(0, 10, nc), rng.uniform(0, 3, nc),
                                 rng.uniform(0.5, 1.5, nc), np.full(nc, 0.3)])
            q = rng.random((nc, 1))
            fb.upload(0, u0)
            sampled, counts = fb.couple(0, c, npm, q)
            ref, s_ref, c_ref = oracle.couple(grid, c, [u0], q)
            assert np.array_equal(counts, c_ref)
            assert np.allclose(sampled, s_ref, rtol=1e-13)
            assert np.allclose(fb.download(0), ref[0], rtol=1e-13)


def test_device_memory_off_the_words(eqf):
    """A device array that starts between two words, in and out."""
    import torch
    nx, ny = 37, 20
    n = (nx + 1) * (ny + 1)
    u = np.random.default_rng(4).random(n)
    raw = torch.zeros(8 * n + 16, dtype=torch.uint8, device="cuda")
    raw[4:4 + 8 * n] = torch.from_numpy(u).view(torch.uint8).cuda()
    torch.cuda.synchronize()
    with eqf.FieldBatch([eqf.field_desc(nx, ny, 3.7, 2.0, 0.1, 100.0)], solver=eqf.solver_desc(eqf.GMG_CG)) as fb:
        fb.upload_dev(0, raw.data_ptr() + 4, n)
        fb.sync()
        assert np.array_equal(fb.download(0), u)
        raw.zero_()
        torch.cuda.synchronize()
        fb.download_dev(0, raw.data_ptr() + 4, n)
        fb.sync()
        assert np.array_equal(raw[4:4 + 8 * n].cpu().view(torch.float64).numpy(), u)
