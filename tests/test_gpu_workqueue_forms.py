"""The workqueue by voxel-column intervals and the shared-ray values of its
pairs against the oracle's serial scan and per-pair rays, bit for bit, over
the forms where they can go wrong: grids of one column, one cell per axis and
more columns than a workgroup, lines along x, z and y, bounded calls that stop
and resume anywhere, and pair lists in and out of channel order."""
import numpy as np
import pytest

from conftest import oracle_geom
from raptr_amd.geometry import MeasurementSetup, VoxelGrid
from test_gpu_rays import CASES

pytestmark = pytest.mark.gpu


def _list(setup, grid, many):
    """Few entries: every voxel is tested.  More than 4,096 tiles of 1,024
    voxels: by column intervals (of grids of 4 cells and more along z)."""
    rng = np.random.default_rng(8)
    if many:
        return rng.integers(0, setup.nchannels, 4096 // (-(-grid.nvox // 1024)) + 9).astype(np.int32)
    return rng.choice(setup.nchannels, min(12, setup.nchannels), replace=False).astype(np.int32)


@pytest.mark.parametrize("many", [False, True], ids=["few", "many"])
@pytest.mark.parametrize("name", ["one_ray", "fine", "ragged", "flat_y", "flat_z", "one_voxel",
                                  "off_centre", "long_x", "long_z", "along_y", "inside",
                                  "same_heads"])
def test_workqueue_forms(gpu, oracle, name, many):
    from raptr_amd import sysmat
    setup, grid, nrays = CASES[name]
    s, g = oracle_geom(oracle, setup, grid)
    lst = _list(setup, grid, many)
    oc, ov, _, _ = oracle.workqueue(s, g, lst)
    c, v, li, vi = sysmat.workqueue(setup, grid, lst)
    np.testing.assert_array_equal(c, oc)
    np.testing.assert_array_equal(v, ov)
    assert (li, vi) == (len(lst), 0)
    np.testing.assert_array_equal(sysmat.workqueue_counts(setup, grid, lst),
                                  oracle.workqueue_counts(s, g, lst))
    # bounded calls of odd lengths, each from where the last one stopped
    li = vi = at = 0
    for n in (1, 7, 300, 1023, 5000, len(ov)):
        n = min(n, len(ov) - at)
        if n == 0:
            break
        c, v, li, vi = sysmat.workqueue(setup, grid, lst, li, vi, n)
        np.testing.assert_array_equal(c, oc[at:at + n])
        np.testing.assert_array_equal(v, ov[at:at + n])
        at += n
    if len(ov) and not many:
        got = sysmat.sm_from_wq(setup, grid, oc, ov, nrays)
        np.testing.assert_array_equal(got, oracle.sm_from_wq(s, g, oc, ov, nrays))


@pytest.mark.parametrize("raygen", ["rand", "regu"])
@pytest.mark.parametrize("length", [1, 255, 1024, 1025, 5000])
@pytest.mark.parametrize("order", ["runs", "six", "seven", "shuffled"])
def test_pair_values_any_order(gpu, oracle, raygen, length, order):
    """Chunks of one channel, of six and seven runs (the last chunk shape with
    shared rays and the first without), of a channel that returns, and of
    channels at random, with pairs outside the setup and the grid."""
    from raptr_amd import sysmat
    setup, grid, nrays = CASES["ragged"]
    s, g = oracle_geom(oracle, setup, grid)
    rg = oracle.RAYGEN_RAND if raygen == "rand" else oracle.RAYGEN_REGU
    rng = np.random.default_rng(length)
    vox = rng.integers(0, grid.nvox, length).astype(np.int32)
    pool = rng.choice(setup.nchannels, 64, replace=False).astype(np.int32)
    pos = np.arange(length)
    cnl = {"runs": pool[pos // 1500 % 64], "six": pool[pos % 1024 * 6 // 1024 % 3],
           "seven": pool[pos % 1024 * 7 // 1024], "shuffled": rng.permutation(
               np.resize(pool, length))}[order].astype(np.int32)
    want = oracle.sm_from_wq(s, g, cnl, vox, nrays, raygen=rg, seed=3)
    np.testing.assert_array_equal(sysmat.sm_from_wq(setup, grid, cnl, vox, nrays, seed=3,
                                                    raygen=rg), want)
    bad = rng.random(length) < 0.2
    cnl[bad] = rng.choice([-1, setup.nchannels, 2**31 - 1], int(bad.sum()))
    vox[~bad & (rng.random(length) < 0.1)] = grid.nvox
    want[bad | (vox == grid.nvox)] = 0
    np.testing.assert_array_equal(sysmat.sm_from_wq(setup, grid, cnl, vox, nrays, seed=3,
                                                    raygen=rg), want)


@pytest.mark.parametrize("name,length", [("ragged", 560001), ("rays_32", 1), ("rays_32", 255),
                                         ("rays_32", 256), ("rays_32", 150001)])
@pytest.mark.parametrize("order", ["runs", "few", "most", "one more", "shuffled"])
def test_pair_values_by_runs(gpu, oracle, name, length, order):
    """Queues whose chunks share a channel's rays: long ones, and short ones of
    many rays; chunks of one run, of as many as share (9 with 9 rays and 74
    planes, 27 with 32 and 51) and of one more."""
    from raptr_amd import sysmat
    setup, grid, nrays = CASES[name]
    s, g = oracle_geom(oracle, setup, grid)
    most = int((7.5 + 9.3 * nrays) / (8 + 0.0018 * nrays * (sum(grid.n) + 3)))
    assert most == {"ragged": 9, "rays_32": 27}[name]
    rng = np.random.default_rng(length)
    vox = rng.integers(0, grid.nvox, length).astype(np.int32)
    pool = rng.choice(setup.nchannels, 64, replace=False).astype(np.int32)
    pos = np.arange(length)
    chunk = min(1024, length)

    def runs(k):
        return pool[(pos // chunk + pos % chunk * k // chunk) % 64]
    cnl = {"runs": pool[pos // 1500 % 64], "few": runs(3), "most": runs(most),
           "one more": runs(most + 1),
           "shuffled": rng.permutation(np.resize(pool, length))}[order].astype(np.int32)
    want = oracle.sm_from_wq(s, g, cnl, vox, nrays, seed=3)
    np.testing.assert_array_equal(sysmat.sm_from_wq(setup, grid, cnl, vox, nrays, seed=3), want)
    bad = rng.random(length) < 0.001
    cnl[bad] = rng.choice([-1, setup.nchannels, 2**31 - 1], int(bad.sum()))
    want[bad] = 0
    np.testing.assert_array_equal(sysmat.sm_from_wq(setup, grid, cnl, vox, nrays, seed=3), want)


@pytest.mark.parametrize("v,o1", [(2.504554271697998, 99406.609375),
                                  (2.5129311084747314, 99405.75),
                                  (2.521639347076416, 99403.3359375)])
def test_coordinates_that_round_coarsely(gpu, oracle, v, o1):
    """Heads 900 mm apart with 20,000 rows of 10 um pixels, in um: the centres
    round by more than a ten-thousandth of the cull's radius, and a voxel
    outside it by FP64 passes the float test."""
    from raptr_amd import sysmat
    ny = 20000
    setup = MeasurementSetup(-450e3, 450e3, 1, 1, ny, 1, ny, 0.0, 10.0, 10.0, 10.0)
    grid = VoxelGrid((-0.5 * v, o1, -1.5 * v), (v, v, v), (1, 200, 4))
    s, g = oracle_geom(oracle, setup, grid)
    c = setup.lin_id(0, ny - 35, 0, ny - 35, 0)
    want = oracle.workqueue(s, g, np.array([c], np.int32))[1]
    lst = np.full(4100, c, np.int32)
    got = sysmat.workqueue(setup, grid, lst)
    np.testing.assert_array_equal(got[1], np.tile(want, len(lst)))
    np.testing.assert_array_equal(sysmat.workqueue_counts(setup, grid, lst), len(want))
    A = sysmat.build_csr(setup, grid, lst[:3], 4, keep_zeros=True).to_host()
    np.testing.assert_array_equal(A[1], np.tile(want, 3))
