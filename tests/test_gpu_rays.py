"""The ray-mask build (zeros dropped, rays per channel) against the oracle,
which tests every culled candidate against every ray: row pointers, columns
and values bit for bit, over the forms where the masks, the rectangles or the
segments can go wrong.  The projections that share the kernel are compared
with FP64 sums over the oracle's matrix (1e-12: FP64 rounding of a few
thousand terms)."""
import numpy as np
import pytest

from conftest import oracle_geom
from raptr_amd.geometry import MeasurementSetup, VoxelGrid, centred_grid, two_head_setup

pytestmark = pytest.mark.gpu

CASES = {
    # one ray; exactly 32 bits; bits shared by 2 and by 3 rays, uneven last run
    "one_ray": (two_head_setup(4, 3, 60.0), centred_grid(16, 5.0), 1),
    "rays_32": (two_head_setup(4, 3, 60.0), centred_grid(16, 5.0), 32),
    "rays_33": (two_head_setup(4, 3, 60.0), centred_grid(16, 5.0), 33),
    "rays_95": (two_head_setup(4, 3, 60.0), centred_grid(16, 5.0), 95),
    # small voxels: ranges wider than the mask words, rows of many segments
    "fine": (two_head_setup(3, 8, 22.5), centred_grid(64, 0.7), 12),
    "ragged": (two_head_setup(5, 7, 25.7), VoxelGrid((-31.0, -7.5, -40.2), (1.9, 2.3, 2.7),
                                                     (37, 5, 29)), 9),
    # grids of one cell on an axis, one voxel, and off the axis
    "flat_y": (two_head_setup(4, 5, 36.0), VoxelGrid((-30.0, -2.0, -30.0), (3.0, 4.0, 3.0),
                                                     (20, 1, 20)), 8),
    "flat_z": (two_head_setup(4, 5, 36.0), VoxelGrid((-30.0, -30.0, -2.0), (3.0, 3.0, 4.0),
                                                     (20, 20, 1)), 8),
    "one_voxel": (two_head_setup(4, 4, 45.0), VoxelGrid((-3.0, -3.0, -3.0), (6.0, 6.0, 6.0),
                                                        (1, 1, 1)), 7),
    "off_centre": (two_head_setup(4, 5, 36.0), VoxelGrid((40.0, -6.0, 10.0), (2.5, 2.5, 2.5),
                                                         (24, 12, 30)), 6),
    # more x cells than a workgroup has threads
    "long_x": (two_head_setup(3, 4, 45.0), VoxelGrid((-150.0, -6.0, -8.0), (1.0, 3.0, 4.0),
                                                     (300, 4, 4)), 8),
    "long_z": (two_head_setup(3, 4, 45.0), VoxelGrid((-8.0, -6.0, -150.0), (4.0, 3.0, 1.0),
                                                     (4, 4, 300)), 8),
    # lines that run mostly along y
    "along_y": (MeasurementSetup(-20.0, 20.0, 3, 2, 24, 2, 24, 60.0, 6.0, 8.0, 4.0),
                centred_grid(20, 4.0), 8),
    # the grid holds the heads: rays start and end inside it
    "inside": (two_head_setup(3, 4, 45.0, pos=30.0), centred_grid(24, 4.0), 8),
    # both heads in one place: rays of any direction, channels without a line
    "same_heads": (MeasurementSetup(5.0, 5.0, 3, 3, 3, 3, 3, 40.0, 20.0, 4.0, 4.0),
                   centred_grid(16, 3.0), 8),
}


def _rows(setup, most=160):
    rng = np.random.default_rng(3)
    k = min(setup.nchannels, most)
    return rng.choice(setup.nchannels, k, replace=False).astype(np.int32)


@pytest.mark.parametrize("regu", [False, True], ids=["rand", "regu"])
@pytest.mark.parametrize("name", list(CASES))
def test_ray_build_is_the_oracles(gpu, oracle, name, regu):
    """REGU rays repeat one line per channel, parallel to an axis for the
    channels of opposite pixels (the slab method then ignores that axis)."""
    from raptr_amd import sysmat
    from raptr_amd.device import DeviceArray
    setup, grid, nrays = CASES[name]
    raygen = oracle.RAYGEN_REGU if regu else oracle.RAYGEN_RAND
    s, g = oracle_geom(oracle, setup, grid)
    lst = _rows(setup)
    if regu:  # opposite pixels of the first angle among them
        d = setup.lin_id(0, 0, 0, 0, 0)
        lst = np.unique(np.append(lst, [d, setup.lin_id(1, 1, 1, 1, 0),
                                        setup.lin_id(1, 0, 0, 0, 0)])).astype(np.int32)
    rp, col, val, _ = oracle.build_csr(s, g, lst, nrays, raygen=raygen, seed=7)
    # the smallest staging area that holds the longest row, too
    for staging in (1 << 16, max(3072, int(np.diff(rp).max())) + 64):
        A = sysmat.build_csr(setup, grid, lst, nrays, raygen=raygen, seed=7, staging=staging)
        grp, gcol, gval = A.to_host()
        np.testing.assert_array_equal(grp, rp)
        np.testing.assert_array_equal(gcol, col)
        np.testing.assert_array_equal(gval, val)
    x = np.random.default_rng(5).random(grid.nvox).astype(np.float32)
    row = np.repeat(np.arange(len(lst)), np.diff(rp))
    fwd = np.bincount(row, val.astype(np.float64) * x[col], len(lst))
    got = sysmat.forward_project(setup, grid, DeviceArray.from_numpy(x), nrays, cnl_list=lst,
                                 raygen=raygen, seed=7)
    np.testing.assert_allclose(got, fwd, rtol=1e-12, atol=1e-12)
    wgt = np.random.default_rng(6).random(len(lst)).astype(np.float32)
    back = np.bincount(col, val.astype(np.float64) * wgt[row], grid.nvox)
    got = sysmat.backproject(setup, grid, nrays, lst, wgt, raygen=raygen, seed=7,
                             normalise=False)
    np.testing.assert_allclose(got, back, rtol=1e-12, atol=1e-12)


def test_ray_build_skips_bad_channels(gpu, oracle):
    """Ids outside the setup give empty rows and no projection."""
    from raptr_amd import sysmat
    from raptr_amd.device import DeviceArray
    setup, grid, nrays = CASES["one_ray"]
    lst = np.array([-1, 3, setup.nchannels, 5], np.int32)
    A = sysmat.build_csr(setup, grid, lst, nrays)
    rp = A.to_host()[0]
    assert rp[1] == rp[0] and rp[3] == rp[2]
    s, g = oracle_geom(oracle, setup, grid)
    orp, _, val, _ = oracle.build_csr(s, g, np.array([3, 5], np.int32), nrays)
    np.testing.assert_array_equal(A.to_host()[2], val)
    got = sysmat.forward_project(setup, grid, DeviceArray.from_numpy(
        np.ones(grid.nvox, np.float32)), nrays, cnl_list=lst)
    assert got[0] == 0 and got[2] == 0


def test_build_kernels_meet(gpu, oracle):
    """Zeros kept runs the candidate build: its non-zero entries are the
    ray-mask build's (a grid whose masks would not fit LDS runs it too)."""
    from raptr_amd import sysmat
    for name in ("fine", "ragged", "along_y"):
        setup, grid, nrays = CASES[name]
        lst = _rows(setup, 60)
        A = sysmat.build_csr(setup, grid, lst, nrays).to_host()
        B = sysmat.build_csr(setup, grid, lst, nrays, keep_zeros=True).to_host()
        nz = B[2] != 0
        np.testing.assert_array_equal(A[1], B[1][nz])
        np.testing.assert_array_equal(A[2], B[2][nz])
    setup = two_head_setup(2, 2, 90.0)
    grid = VoxelGrid((-200.0, -4.0, -4.0), (0.16, 4.0, 4.0), (2500, 2, 2))
    lst = np.arange(setup.nchannels, dtype=np.int32)
    s, g = oracle_geom(oracle, setup, grid)
    rp, col, val, _ = oracle.build_csr(s, g, lst, 4)
    got = sysmat.build_csr(setup, grid, lst, 4).to_host()
    for a, b in zip(got, (rp, col, val)):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("staging", [1 << 14, 1 << 17, 1 << 19])
def test_staging_areas(gpu, oracle, staging):
    """Lists whose chunks reach the 64 staging areas (1,024 rows) and overflow
    them: rows outside the grid, then long rows, then rows of both kinds."""
    from raptr_amd import sysmat
    setup, grid = two_head_setup(6, 5, 36.0), centred_grid(24, 0.5)
    s, g = oracle_geom(oracle, setup, grid)
    every = np.arange(setup.nchannels, dtype=np.int32)
    n = np.diff(oracle.build_csr(s, g, every, 6, seed=3)[0])
    order = np.argsort(n, kind="stable").astype(np.int32)
    rng = np.random.default_rng(2)
    lst = np.concatenate([order[:3000], order[-1500:], rng.permutation(order)]).astype(np.int32)
    assert n[order[:1500]].max() == 0 and n[order[-1500:]].min() >= 160
    rp, col, val, _ = oracle.build_csr(s, g, lst, 6, seed=3)
    A = sysmat.build_csr(setup, grid, lst, 6, seed=3, staging=staging)
    for got, want in zip(A.to_host(), (rp, col, val)):
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("nz", [387, 388, 394])
def test_candidate_build_at_the_lds_limit(gpu, oracle, nz):
    """70 rays: the candidate build's tables with its own arrays leave a CU's 160
    KiB from 395 planes on, the tables alone beyond 401.  It is refused there; the
    ray masks, which need less, are not."""
    from raptr_amd import sysmat
    from raptr_amd import _capi as capi
    setup, grid = two_head_setup(2, 2, 90.0), VoxelGrid((-4.0, -4.0, -97.0), (4.0, 4.0, 0.5),
                                                        (2, 2, nz))
    lst = np.arange(setup.nchannels, dtype=np.int32)
    s, g = oracle_geom(oracle, setup, grid)
    rp, col, val, _ = oracle.build_csr(s, g, lst, 70)
    for got, want in zip(sysmat.build_csr(setup, grid, lst, 70).to_host(), (rp, col, val)):
        np.testing.assert_array_equal(got, want)
    if nz == 387:
        A = sysmat.build_csr(setup, grid, lst, 70, keep_zeros=True).to_host()
        np.testing.assert_array_equal(A[2][A[2] != 0], val)
    else:
        for kw in (dict(keep_zeros=True), dict(raygen=capi.RAYGEN_RAND_ELEMENT)):
            with pytest.raises(capi.RaptrError) as e:
                sysmat.build_csr(setup, grid, lst, 70, **kw)
            assert e.value.status == capi.RAPTR_ERR_NOT_SUPPORTED
