"""The parallel affine coupling (overlap rows, triangular solve, tile deposit)
where it can go wrong: a chain of overlaps across the solve's 1024-cell chunk,
more overlaps than a cell has slots for (the sequential walk takes the call),
centre-node cells on one node, traps without cells, species counts at the edges
of a pass.  The oracle's sequential loop is the reference: counts exact;
samples within 1e-13 relative (sums of at most 600 nodes, 6.6e-14) and fields
within 1e-14 (each node a handful of additions), as the existing affine test."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NPM = 10.0


def _row(n, step, y):
    c = np.zeros((n, 5))
    c[:, 0] = 2.0 + step * np.arange(n)
    c[:, 1], c[:, 3], c[:, 4] = y, 3.0, 1.0
    return c


def _cells(kind, rng):
    """(nx, ny, cells) of each trap."""
    few = np.column_stack([rng.uniform(0, 12, 40), rng.uniform(0, 6, 40), rng.uniform(0, 3, 40),
                           rng.uniform(2, 4, 40), np.ones(40)])
    if kind == "chain":
        return [(5560, 30, _row(1100, 0.5, 1.53)), (120, 60, few)]
    if kind == "stack":  # 40 rods on one place: over the 32 slots
        c = few.copy()
        c[:, :2] = 5.03, 3.04
        return [(120, 60, few), (120, 60, c)]
    if kind == "points":  # boxes that hold no node: the centre node of each, ten cells a node
        c = few.copy()
        c[:, 0] = 1.0 + 0.1 * (np.arange(40) // 10) + 0.03
        c[:, 1], c[:, 3], c[:, 4] = 1.04, 0.03, 0.02
        return [(120, 60, c), (120, 60, few[:0]), (120, 60, few[:1])]
    return [(120, 60, few), (120, 60, few[::-1].copy())]


@pytest.mark.parametrize("kind,ns", [("chain", 2), ("stack", 2), ("points", 1), ("few", 4), ("few", 5)])
def test_affine_coupling(eqf, oracle, kind, ns):
    import torch
    from eq_amd import workloads as Wl
    rng = np.random.default_rng(5)
    traps = _cells(kind, rng)
    off = np.concatenate([[0], np.cumsum([c.shape[0] for _, _, c in traps])]).astype(np.int64)
    a = rng.uniform(0.05, 0.15, (off[-1], ns))
    b = -0.05 * rng.uniform(0.5, 1.0, (off[-1], ns))
    descs = [eqf.field_desc(nx, ny, nx / NPM, ny / NPM, 0.1, 200.0, 0.01, 0.0, Wl.TOP_DIRICHLET)
             for nx, ny, _ in traps for _ in range(ns)]
    u0 = [rng.random((d.nx + 1) * (d.ny + 1)) for d in descs]
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    cells_d, a_d, b_d = dev(np.concatenate([c for _, _, c in traps])), dev(a), dev(b)
    samp_d = torch.zeros((int(off[-1]), ns), dtype=torch.float64, device="cuda")
    cnt_d = torch.zeros(int(off[-1]), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    with eqf.FieldBatch(descs, nspecies=ns, solver=eqf.solver_desc(eqf.MIXED_GMG_CG)) as fb:
        for _ in range(2):  # the second call has its buffers sized from the first
            for k, u in enumerate(u0):
                fb.upload(k, u)
            fb.couple_affine_dev(0, off, cells_d.data_ptr(), NPM, a_d.data_ptr(), b_d.data_ptr(), samp_d.data_ptr(),
                                 cnt_d.data_ptr())
            fb.sync()
            samp, cnt = samp_d.cpu().numpy(), cnt_d.cpu().numpy()
            for t, (nx, ny, c) in enumerate(traps):
                if not len(c):
                    continue
                at = slice(off[t], off[t + 1])
                grid = oracle.grid(nx + 1, ny + 1, NPM, nx / NPM, ny / NPM)
                fields, s_ref, c_ref = oracle.couple_affine(grid, c, u0[ns * t:ns * t + ns], a[at], b[at])
                assert np.array_equal(cnt[at], c_ref)
                assert np.allclose(samp[at], s_ref, rtol=1e-13, atol=1e-300)
                for s in range(ns):
                    assert np.allclose(fb.download(ns * t + s), fields[s], rtol=1e-14, atol=1e-15), (t, s)


@pytest.mark.parametrize("near", [80, 96, 97, 130])
def test_affine_coupling_windows_without_overlaps(eqf, oracle, monkeypatch, near):
    """A long rod whose window meets those of `near` small cells beside it, none
    of which it covers: on both sides of the windows a cell may meet (96)."""
    x, y = np.meshgrid(np.arange(2.2, 9.8, 0.3), np.arange(0.9, 5.1, 0.3))
    away = np.abs(0.447 * (x - 6.0) - 0.894 * (y - 3.0)) > 0.9
    c = np.zeros((near + 1, 5))
    c[:near, 0], c[:near, 1] = x[away][:near] + 0.01, y[away][:near] + 0.01
    c[:near, 3], c[:near, 4] = 0.15, 0.1
    c[near] = 6.0, 3.0, 0.4636, 10.0, 1.0
    monkeypatch.setattr(sys.modules[__name__], "_cells", lambda kind, rng: [(120, 60, c), (120, 60, c[:3])])
    test_affine_coupling(eqf, oracle, "windows", 2)


def test_affine_coupling_without_room_for_its_rows(eqf, oracle):
    """A million cells on a device with 250 MiB left: the geometry fits (130 MB),
    the overlap rows (256 MB) do not, and the walk in list order takes the call.
    Samples within 1e-12: sums of 300 nodes in another order, 3e-14, carried on
    by amounts that depend on them."""
    import torch
    rng = np.random.default_rng(9)
    nx, ny, n = 1000, 500, 1000000
    cells = np.column_stack([rng.uniform(0, nx / NPM, n), rng.uniform(0, ny / NPM, n), rng.uniform(0, 3, n),
                             rng.uniform(2, 4, n), np.ones(n)])
    a, b, u0 = rng.uniform(0.05, 0.15, (n, 1)), -0.05 * rng.uniform(0.5, 1.0, (n, 1)), rng.random((nx + 1) * (ny + 1))
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    cells_d, a_d, b_d = dev(cells), dev(a), dev(b)
    samp_d = torch.zeros((n, 1), dtype=torch.float64, device="cuda")
    cnt_d = torch.zeros(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    with eqf.FieldBatch([eqf.field_desc(nx, ny, nx / NPM, ny / NPM, 0.1, 200.0)], solver=eqf.solver_desc(eqf.GMG_CG)) as fb:
        def couple(k):
            fb.couple_affine_dev(0, np.array([0, k], np.int64), cells_d.data_ptr(), NPM, a_d.data_ptr(), b_d.data_ptr(),
                                 samp_d.data_ptr(), cnt_d.data_ptr())
            fb.sync()
        couple(100)  # the kernels and the tables of a first call
        fb.upload(0, u0)
        room = [torch.empty(50 << 20, dtype=torch.uint8, device="cuda") for _ in range(5)]
        filler, size = [], 1 << 36
        while size >= 10 << 20:  # until nothing of 10 MiB is left
            try:
                filler.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                size //= 2
        del room
        torch.cuda.empty_cache()
        try:
            couple(n)
        finally:
            del filler
            torch.cuda.empty_cache()
        fields, s_ref, c_ref = oracle.couple_affine(oracle.grid(nx + 1, ny + 1, NPM, nx / NPM, ny / NPM), cells, [u0], a, b)
        assert np.array_equal(cnt_d.cpu().numpy(), c_ref)
        assert np.allclose(samp_d.cpu().numpy(), s_ref, rtol=1e-12)
        assert np.allclose(fb.download(0), fields[0], rtol=1e-12)
