"""The ends of an iteration and the shapes that depend on a plan's size, on
both sides of each rule: the one-pass and the per-XCD column reduce of the
fused iteration's mode 1, the normalisation in one launch and in two, runs of
iterations per graph replay, the 64-frame forward with a group per workgroup
and per wave, and the 64-frame reduce over several voxels.  References: the
FP64 recurrence on the plan's matrix (1e-5: FP32 sums of a few hundred terms
over five iterations, measured by the plan's other tests at 1e-6) and other
shapes of the same plan (1e-6, FP32 summation order)."""
import numpy as np
import pytest

from raptr_amd.geometry import VoxelGrid, centred_grid, two_head_setup

pytestmark = pytest.mark.gpu


def _system(setup, grid, nrays, rows=None, seed=1):
    from raptr_amd import sysmat
    from raptr_amd.device import DeviceArray
    rng = np.random.default_rng(seed)
    lst = np.arange(setup.nchannels, dtype=np.int32)
    if rows:
        lst = np.sort(rng.choice(lst, rows, replace=False)).astype(np.int32)
    A = sysmat.build_csr(setup, grid, lst, nrays)
    rp, col, val = A.to_host()
    val = val.astype(np.float64)
    row = np.repeat(np.arange(A.m), np.diff(rp))
    sens = np.bincount(col, val, grid.nvox)
    x = np.zeros(grid.nvox)
    x[rng.choice(grid.nvox, grid.nvox // 3, replace=False)] = rng.random(grid.nvox // 3)
    yb = np.bincount(row, val * x[col], A.m)
    y = rng.poisson(yb * (20.0 / max(yb.max(), 1e-30))).astype(np.float32)
    return A, DeviceArray.from_numpy(sens), sens, (row, col, val), y


def _mlem64(mat, m, n, y, sens, niter):
    row, col, val = mat
    s = sens / sens.sum()
    s = s + (s == 0)
    x = np.full(n, 1.0 / n)
    for _ in range(niter):
        yt = np.bincount(row, val * x[col], m)
        e = np.divide(y.astype(np.float64), yt, out=np.zeros(m), where=yt != 0)
        x = x * np.bincount(col, val * e[row], n) / s
        x /= x.sum()
    return x


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _x0(n):
    return np.full(n, 1.0 / n, np.float32)


@pytest.mark.parametrize("grid,split", [(centred_grid(12, 6.0), True),
                                        (centred_grid(32, 2.5), False)])
def test_mode1_reduce_both_forms(gpu, grid, split):
    """Many (12^3) and few (32^3) union entries per column: mode 1 splits
    the columns by XCD or takes them in one pass."""
    from raptr_amd.recon import Reconstructor
    setup = two_head_setup(8, 25 if split else 5, 7.2 if split else 36.0)
    A, dsens, sens, mat, y = _system(setup, grid, 10)
    R = Reconstructor(A, dsens, "f32", 1, row_order=setup)
    R.set_union_rows(16)
    u = R.unions()
    assert R.fused()["available"] and (u["entries"] >= 128 * grid.nvox) == split
    want = _mlem64(mat, A.m, grid.nvox, y, sens, 5)
    images = []
    for mode in (1, 0):
        R.set_fused_reduce(mode)
        images.append(R.mlem(y, _x0(grid.nvox), 5))
        assert _rel(images[-1], want) <= 1e-5
        np.testing.assert_array_equal(R.mlem(y, _x0(grid.nvox), 5), images[-1])
    assert _rel(images[0], images[1]) <= 1e-6


@pytest.mark.parametrize("grid", [VoxelGrid((-66.0, -64.4, -65.2), (0.8, 0.8, 0.8), (165, 161, 163)),
                                  centred_grid(17, 5.0)], ids=["2 launches", "1 launch"])
def test_normalisation_launches(gpu, grid):
    """More than 16,384 partial sums (4.33M voxels) and fewer."""
    from raptr_amd.recon import Reconstructor
    setup = two_head_setup(6, 5, 36.0)
    A, dsens, sens, mat, y = _system(setup, grid, 6, rows=700)
    for order in (setup, None):  # fused iteration, separate passes
        R = Reconstructor(A, dsens, "f32", 1, row_order=order)
        if order is None:
            R.set_fused(False)
        x = R.mlem(y, _x0(grid.nvox), 5)
        assert _rel(x, _mlem64(mat, A.m, grid.nvox, y, sens, 5)) <= 1e-5
        assert abs(float(x.astype(np.float64).sum()) - 1.0) <= 1e-5
        R.close()


def test_graph_runs_equal_eager(gpu):
    """Replays of one iteration and of four at a time give the eager
    images, interleaved with eager runs, and share one cache entry."""
    from raptr_amd.device import DeviceArray, Stream
    from raptr_amd.recon import Reconstructor
    setup, grid = two_head_setup(4, 6, 30.0), centred_grid(16, 5.0)
    A, dsens, _, _, y = _system(setup, grid, 6)
    st = Stream()
    for F in (1, 64):
        R = Reconstructor(A, dsens, "f32", F, row_order=setup, grid=grid, stream=st.handle)
        Y = np.repeat(y[:, None], F, axis=1).reshape(-1)
        X0 = np.repeat(_x0(grid.nvox)[:, None], F, axis=1).reshape(-1)
        dy = DeviceArray.from_numpy(Y, stream=st.handle)
        dx = DeviceArray(grid.nvox * F, np.float32)
        for niter in (2, 3, 4, 5, 9, 4, 2, 13):
            dx.copy_from(X0, stream=st.handle)
            R.run(dy, dx, niter, F, use_graph=False, stream=st.handle)
            eager = dx.numpy(stream=st.handle)
            dx.copy_from(X0, stream=st.handle)
            R.run(dy, dx, niter, F, use_graph=True, stream=st.handle)
            np.testing.assert_array_equal(dx.numpy(stream=st.handle), eager)
        from raptr_amd import _capi as capi
        assert capi.lib().raptr_recon_graph_count(R.handle) == 1
        R.close()


@pytest.mark.parametrize("rows,grid", [(131072, centred_grid(7, 12.0)), (131089, centred_grid(7, 12.0)),
                                       (33, VoxelGrid((-49.5, -34.1, -57.2), (2.2, 2.2, 2.2), (45, 31, 52))),
                                       (17, centred_grid(5, 16.0))])
@pytest.mark.parametrize("vt", ["f32", "f16"])
def test_frames64_both_forwards(gpu, rows, grid, vt):
    """8,192 row groups and one more, ragged row and voxel counts, fewer rows
    than a block of 16 for each XCD: 64 frames against single frames."""
    from raptr_amd.recon import Reconstructor
    setup = two_head_setup(13, 5, 36.0)
    A, dsens, _, _, y = _system(setup, grid, 4, rows=rows)
    R = Reconstructor(A, dsens, vt, 64, row_order=setup, grid=grid)
    assert R.grouped()["on"] == 1
    rng = np.random.default_rng(4)
    Y = np.repeat(y[:, None], 64, axis=1)
    Y[:, 1:] *= rng.integers(0, 3, (A.m, 63)).astype(np.float32)
    Y[:, 63] = 0.0  # an empty frame stays finite
    X = R.mlem(Y, np.repeat(_x0(grid.nvox)[:, None], 64, axis=1), 4)
    R.close()
    R1 = Reconstructor(A, dsens, vt, 1, row_order=setup)
    for f in (0, 1, 31, 62):
        assert _rel(X[:, f], R1.mlem(np.ascontiguousarray(Y[:, f]), _x0(grid.nvox), 4)) <= 1e-6
    assert np.all(X[:, 63] == 0.0)


@pytest.mark.parametrize("rows", [20011, 131089], ids=["split lists", "a wave a group"])
@pytest.mark.parametrize("vt", ["f32", "f16", "bf16", "u16"])
def test_frames64_every_forward_shape(gpu, rows, vt):
    """Both forwards with each unroll, kind and number of active frames.  The
    unroll is what the forward runs: with split lists it moves the cuts between
    the waves, so some sums round otherwise."""
    from raptr_amd import _capi as capi
    from raptr_amd.device import DeviceArray
    from raptr_amd.recon import Reconstructor
    grid = centred_grid(7, 12.0)
    A, dsens, _, _, y = _system(two_head_setup(13, 5, 36.0), grid, 4, rows=rows)
    R = Reconstructor(A, dsens, vt, 64, row_order=two_head_setup(13, 5, 36.0), grid=grid)
    split = (rows + 15) // 16 <= 8192
    assert R.grouped()["unroll"] == (16 if split else 8)
    Y = np.repeat(y[:, None], 64, axis=1)
    Y[:, 1:] *= np.random.default_rng(4).integers(1, 4, (A.m, 63)).astype(np.float32)
    X0 = np.repeat(_x0(grid.nvox)[:, None], 64, axis=1)
    base = R.mlem(Y, X0, 3)
    dy, ratios = DeviceArray.from_numpy(Y.reshape(-1)), {}
    de = DeviceArray(A.m * 64, np.float32)
    for unroll, kind in Reconstructor.GROUP_SHAPES[16]:
        R.set_grouped(True, unroll, kind)
        X = R.mlem(Y, X0, 3)
        assert _rel(X, base) <= 1e-6, (unroll, kind)
        for active in (16, 32) if kind == 3 else ():
            dx = DeviceArray.from_numpy(X0.reshape(-1))
            R.run(dy, dx, 3, 64, use_graph=False, active=active)
            np.testing.assert_array_equal(dx.numpy().reshape(grid.nvox, 64)[:, :active],
                                          X[:, :active], err_msg=f"{unroll} {kind} {active}")
        dx = DeviceArray.from_numpy(base.reshape(-1))
        capi.call("raptr_recon_forward", R.handle, 64, dx.ptr, dy.ptr, de.ptr, None)
        ratios[unroll] = de.numpy()
    for unroll in (16, 32):
        assert _rel(ratios[unroll], ratios[8]) <= 1e-6
    if split:
        assert (ratios[32] != ratios[8]).any()
    R.close()


@pytest.mark.parametrize("n", [(64, 48, 49), (72, 66, 64), (96, 97, 64)])
def test_frames64_few_ranges(gpu, n):
    """Grids of 9,408, 19,008 and 37,248 bricks under few rows: the backward
    splits its rows in 4, 2 and 1 ranges.  The first 16 frames alone get the
    full pass's images."""
    from raptr_amd.device import DeviceArray
    from raptr_amd.recon import Reconstructor
    setup = two_head_setup(6, 8, 22.5)
    grid = VoxelGrid(tuple(-0.5 * k for k in n), (1.0, 1.0, 1.0), n)
    A, dsens, _, _, y = _system(setup, grid, 5, rows=601)
    R = Reconstructor(A, dsens, "f32", 64, row_order=setup, grid=grid)
    Y = np.repeat(y[:, None], 64, axis=1)
    Y[:, 1:] *= np.random.default_rng(6).integers(1, 4, (A.m, 63)).astype(np.float32)
    X0 = np.repeat(_x0(grid.nvox)[:, None], 64, axis=1)
    X = R.mlem(Y, X0, 4)
    dy, dx = DeviceArray.from_numpy(Y.reshape(-1)), DeviceArray.from_numpy(X0.reshape(-1))
    R.run(dy, dx, 4, 64, use_graph=False, active=16)
    np.testing.assert_array_equal(dx.numpy().reshape(grid.nvox, 64)[:, :16], X[:, :16])
    R.close()
    R1 = Reconstructor(A, dsens, "f32", 1, row_order=setup)
    for f in (0, 15, 40, 63):
        want = R1.mlem(np.ascontiguousarray(Y[:, f]), _x0(grid.nvox), 4)
        assert _rel(X[:, f], want) <= 1e-6
