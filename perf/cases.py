"""Measured workloads of the reconstruction path.

Each case is one call sequence that a user's program makes through the
public entry points of ``raptr_amd`` (the Python package, and the C ABI
through ``_capi`` where a program holds device buffers):

* ``workqueue``: the two-stage path of one chunk of the measurement list
  (raptr_workqueue, then raptr_sm_from_wq on its pairs);
* ``build``: the system matrix of a measurement list into buffers that the
  program holds (raptr_sm_build_csr_ex; with a count call first, or straight
  into buffers of a known bound);
* ``sens``: the FP64 sensitivity image over all channels of a scanner;
* ``project``: one matrix-free projection and the summed back-projection of
  a measurement list (the ``backprojection`` driver's computation);
* ``recon``: MLEM iterations of one frame or a batch of frames on a plan;
* ``reco``: the whole reconstruction of a measurement list, as the ``reco``
  driver runs it between its files: matrix, plan, iterations, image.

Sizes are those of the named configurations (8x8 heads / 32^3, 13x13 heads /
180 angles / 52^3), the serving geometries (up to 16x16 heads / 96^3) and
odd ones between them.  Counts are Poisson draws whose means are line
integrals through a phantom of random ellipsoids on a weak background,
computed here in closed form, so the inputs depend on the seed alone.
"""
import ctypes
import math

import numpy as np
import torch

from raptr_amd import _capi as capi
from raptr_amd import sysmat
from raptr_amd.device import DeviceArray, Stream, Workspace
from raptr_amd.geometry import VoxelGrid, two_head_setup
from raptr_amd.recon import Reconstructor


def listed():
    return [
        # a first chunk of the measurement list through the reference's
        # two-stage interface, small scanner
        dict(name="workqueue_32", kind="workqueue", npix=8, na=5, nx=32, ny=32, nz=32, pitch=2.5,
             nrays=10, channels=3000),
        # the small configuration's matrix over all of its 20,480 channels:
        # counted first, then filled
        dict(name="build_32", kind="build", npix=8, na=5, nx=32, ny=32, nz=32, pitch=2.5,
             nrays=10, channels=20480, count=True),
        # part of the full-size configuration's measurement list
        dict(name="build_52", kind="build", npix=13, na=180, nx=52, ny=52, nz=52, pitch=2.0,
             nrays=30, channels=100003, count=False),
        # the largest serving geometry, a low-count request's list
        dict(name="build_96", kind="build", npix=16, na=60, nx=96, ny=96, nz=96, pitch=2.0,
             nrays=20, channels=20011, count=False),
        # a new scanner's sensitivity image (all 147,456 channels)
        dict(name="sens_32", kind="sens", npix=8, na=36, nx=32, ny=32, nz=32, pitch=2.5,
             nrays=10),
        # simulation and quick-look back-projection of one measurement list,
        # grid with three different edges
        dict(name="project_odd", kind="project", npix=11, na=37, nx=45, ny=31, nz=52, pitch=2.2,
             nrays=17, channels=40009),
        # the smallest reconstruction: 5 iterations of the small
        # configuration, where launches count
        dict(name="recon_32", kind="recon", npix=8, na=5, nx=32, ny=32, nz=32, pitch=2.5,
             nrays=10, events=200000, frames=1, value_type="f32", niter=5),
        # the full-size configuration at a clinical count level (about a
        # million measured channels), 50 iterations
        dict(name="recon_52", kind="recon", npix=13, na=180, nx=52, ny=52, nz=52, pitch=2.0,
             nrays=30, events=2000000, frames=1, value_type="f32", niter=50),
        # large image, 16-bit matrix values, ragged edges
        dict(name="recon_96_u16", kind="recon", npix=16, na=60, nx=96, ny=95, nz=93, pitch=2.0,
             nrays=20, events=300000, frames=1, value_type="u16", niter=20),
        # 64 dynamic frames on the small geometry
        dict(name="frames64_32", kind="recon", npix=8, na=5, nx=32, ny=32, nz=32, pitch=2.5,
             nrays=10, events=200000, frames=64, value_type="f32", niter=30),
        # 64 dynamic frames on the full-size grid
        dict(name="frames64_52", kind="recon", npix=13, na=180, nx=52, ny=52, nz=52, pitch=2.0,
             nrays=30, events=400000, frames=64, value_type="f32", niter=20),
        # a whole reconstruction from the measurement list to the image
        dict(name="reco_52", kind="reco", npix=13, na=120, nx=52, ny=52, nz=52, pitch=2.0,
             nrays=20, events=90000, value_type="f32", niter=30),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["workqueue", "build", "build", "sens", "project", "recon", "recon",
                       "recon", "reco"])
    npix = rng.randint(4, 16 if kind in ("build", "recon") else 13)
    n = _log_int(rng, 16, 96 if kind in ("build", "recon") else 52)
    edges = [n] * 3 if rng.random() < 0.5 else [max(8, n - rng.randint(0, n // 3))
                                               for _ in range(3)]
    case = dict(kind=kind, npix=npix, na=_log_int(rng, 3, 180), nx=edges[0], ny=edges[1],
                nz=edges[2], pitch=rng.choice([2.0, 2.2, 2.5]), nrays=rng.randint(5, 30))
    # scanners of at most the full-size configuration's channels
    case["na"] = max(3, min(case["na"], (5200000 if n <= 52 else 2000000) // npix ** 4))
    if kind == "workqueue":
        case["channels"] = _log_int(rng, 100, 3000)
    elif kind == "build":
        case["channels"] = _log_int(rng, 500, 100000 if n <= 52 else 20000)
        case["count"] = rng.random() < 0.3
    elif kind == "sens":
        most = 147456 * 320 / (case["nrays"] * n)
        case["na"] = max(3, min(case["na"], int(most) // npix ** 4))
    elif kind == "project":
        case["channels"] = _log_int(rng, 500, 40000)
    elif kind == "recon":
        case["frames"] = rng.choice([1, 1, 8, 64])
        case["events"] = _log_int(rng, 10000, 2000000 if case["frames"] == 1 and n <= 52
                                  else 200000 if n <= 52 else 100000)
        case["value_type"] = rng.choice(["f32", "f32", "f32", "u16", "f16"])
        case["niter"] = rng.randint(5, 20)
    else:
        case["events"] = _log_int(rng, 5000, 90000)
        case["value_type"] = "f32"
        case["niter"] = rng.randint(10, 30)
    return case


# ------------------------------------------------------------------ inputs
def _setup(case):
    # heads 460 mm apart, 4 x 4 x 20 mm pixels, na steps over 180 degrees
    return two_head_setup(case["npix"], case["na"], 180.0 / case["na"])


def _grid(case):
    n, p = (case["nx"], case["ny"], case["nz"]), case["pitch"]
    return VoxelGrid(tuple(-0.5 * k * p for k in n), (p, p, p), n)


def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 8191 + stream)
    return g


def _lines(setup, channels):
    """Pixel-centre end points [k, 3] of the channels, FP64."""
    c = channels.to(torch.int64)
    y1 = c % setup.n1y
    c = c // setup.n1y
    z1 = c % setup.n1z
    c = c // setup.n1z
    y0 = c % setup.n0y
    c = c // setup.n0y
    z0 = c % setup.n0z
    a = (c // setup.n0z).double() * (setup.da * math.pi / 180.0)
    ends = []
    for pos, iy, iz, ny, nz in ((setup.pos0x, y0, z0, setup.n0y, setup.n0z),
                                (setup.pos1x, y1, z1, setup.n1y, setup.n1z)):
        py = (iy.double() - 0.5 * (ny - 1)) * setup.segy
        pz = (iz.double() - 0.5 * (nz - 1)) * setup.segz
        ends.append(torch.stack([a.cos() * pos + a.sin() * pz, py,
                                 -a.sin() * pos + a.cos() * pz], 1))
    return ends


def _phantom(setup, grid, seed):
    """Line integrals [7, channels] of all channels through six ellipsoids
    (semi-axes 5-25 mm) and a box over the grid, and the parts' (activity,
    half-life in frames): 0.5-8 and 10-120, 0.1 for the box."""
    rng = np.random.default_rng([int(seed), 77])
    extent = np.array(grid.d) * np.array(grid.n)
    p0, p1 = _lines(setup, torch.arange(setup.nchannels, device="cuda"))
    u = p1 - p0
    length = u.norm(dim=1)
    half = torch.tensor(0.5 * extent, device="cuda")
    t = torch.stack([(-half - p0) / u, (half - p0) / u])
    parts = [length * (t.amax(0).amin(1) - t.amin(0).amax(1)).clamp(0)]
    act, life = [0.1], [math.inf]
    for _ in range(6):
        centre = torch.tensor(rng.uniform(-0.3, 0.3, 3) * extent, device="cuda")
        axes = torch.tensor(rng.uniform(5.0, 25.0, 3), device="cuda")
        act.append(math.exp(rng.uniform(math.log(0.5), math.log(8.0))))
        life.append(rng.uniform(10.0, 120.0))
        q, d = (p0 - centre) / axes, u / axes
        a, b, c = (d * d).sum(1), (q * d).sum(1), (q * q).sum(1) - 1.0
        parts.append(length * 2.0 * (b * b - a * c).clamp(0).sqrt() / a)
    return torch.stack(parts).nan_to_num(0.0), np.array(act), np.array(life)


def _mean_counts(parts, act, life, frame=0.0):
    """Expected counts up to a factor, activities decayed to the frame."""
    return (parts * torch.tensor(act * 0.5 ** (frame / life), device="cuda")[:, None]).sum(0)


def _counts(case, setup, grid, seed):
    """(measured channels int32, counts float32 [m] or [m, F]) as tensors."""
    frames = case.get("frames", 1)
    parts, act, life = _phantom(setup, grid, seed)
    mean = _mean_counts(parts, act, life)
    g = _generator(seed, 1)
    first = torch.poisson(mean * (case["events"] / mean.sum()), generator=g)
    meas = first.nonzero().flatten()
    y = first[meas].float()
    if frames > 1:
        # dynamic frames on the first frame's channels, totals falling to a
        # twentieth
        cols, parts = [y], parts[:, meas]
        for f in range(1, frames):
            lam = _mean_counts(parts, act, life, float(f))
            total = case["events"] * 0.05 ** (f / (frames - 1))
            cols.append(torch.poisson(lam * (total / lam.sum()), generator=g).float())
        y = torch.stack(cols, 1).contiguous()
    return meas.int(), y


def _list(case, setup, grid, seed):
    """A measurement list of case["channels"] channels that see the object,
    ascending; their counts."""
    mean = _mean_counts(*_phantom(setup, grid, seed))
    key = torch.rand(setup.nchannels, generator=_generator(seed, 2), device="cuda",
                     dtype=torch.float64)
    k = min(case["channels"], setup.nchannels)
    pick = (key.log() / mean.clamp(min=1e-30)).topk(k).indices.sort().values
    y = 1.0 + torch.poisson(3.0 * mean[pick] / mean.max(), generator=_generator(seed, 3))
    return pick.int(), y.float()


_sens = {}


def _sensitivity(case, setup, grid):
    """The scanner's sensitivity image on the host.  A site computes it once
    per scanner and grid and keeps it as a file, so it is kept here too."""
    key = (setup, grid, case["nrays"])
    if key not in _sens:
        _sens[key] = sysmat.sensitivity(setup, grid, case["nrays"]).numpy()
    return _sens[key]


class _Span:
    """A device range that torch can wrap."""

    def __init__(self, owner, ptr, shape, dtype):
        self.owner, self.ptr = owner, int(ptr)
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": np.dtype(dtype).str,
                                         "data": (int(ptr), False), "version": 2}


def _tensor(a, shape=None):
    """The elements of a DeviceArray as a torch tensor (no copy)."""
    shape = (a.count,) if shape is None else shape
    if 0 in shape:
        return torch.empty(shape, device="cuda")
    return torch.as_tensor(_Span(a, a.ptr, shape, a.dtype), device="cuda")


def _device_array(t):
    """A DeviceArray with a tensor's values."""
    return DeviceArray.from_numpy(t.cpu().numpy().reshape(-1))


def prepare(case, seed):
    setup, grid, kind = _setup(case), _grid(case), case["kind"]
    s = {"case": case, "setup": setup, "grid": grid, "kind": kind, "nrays": case["nrays"],
         "seed": int(seed) & 0x7fffffff, "stream": Stream()}
    st = s["stream"].handle
    if kind == "sens":
        return s
    if kind in ("workqueue", "build", "project"):
        meas, y = _list(case, setup, grid, seed)
        s["list"] = meas.cpu().numpy()
        s["d_list"] = DeviceArray.from_numpy(s["list"])
        if kind == "project":
            s["counts"] = y.cpu().numpy()
            s["image"] = torch.rand(grid.nvox, generator=_generator(seed, 4),
                                    device="cuda").cpu().numpy()
            return s
        g = ctypes.byref(grid.struct())
        m, cap = len(s["list"]), _capacity(case)
        s["val"] = DeviceArray.zeros(cap, np.float32)
        s["vxl"] = DeviceArray.zeros(cap, np.int32)
        if kind == "workqueue":
            s["cnl"] = DeviceArray.zeros(cap, np.int32)
            s["ws"] = Workspace(capi.lib().raptr_workqueue_workspace_size(g, m))
        if kind == "build":
            s["row_ptr"] = DeviceArray.zeros(m + 1, np.int64)
            s["ws"] = Workspace(capi.lib().raptr_sm_build_workspace_size(
                g, case["nrays"], sysmat.DEFAULT_STAGING))
        return s
    meas, y = _counts(case, setup, grid, seed)
    s["sens"] = DeviceArray.from_numpy(_sensitivity(case, setup, grid))
    if kind == "reco":
        s["list"], s["counts"] = meas.cpu().numpy(), y.cpu().numpy()
        return s
    frames = case["frames"]
    lst = meas.cpu().numpy()
    # one system matrix per scanner: the rays keep one seed
    A = sysmat.build_csr(setup, grid, lst, case["nrays"], seed=1, stream=st, capacity="auto")
    s["plan"] = Reconstructor(A, s["sens"], case["value_type"], frames, stream=st,
                              row_order=setup, grid=grid)
    s["y"] = _device_array(y)
    s["x0"] = DeviceArray.from_numpy(np.full(grid.nvox * frames, 1.0 / grid.nvox, np.float32))
    s["x"] = DeviceArray(grid.nvox * frames, np.float32)
    return s


# ------------------------------------------------------------------- a pass
def run(s):
    setup, grid, kind, nrays, seed = s["setup"], s["grid"], s["kind"], s["nrays"], s["seed"]
    st, case = s["stream"].handle, s["case"]
    su, g = ctypes.byref(setup.struct()), ctypes.byref(grid.struct())
    if kind == "workqueue":
        li, vi, found = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int64()
        capi.call("raptr_workqueue", su, g, s["d_list"].ptr, len(s["list"]), ctypes.byref(li),
                  ctypes.byref(vi), -1, s["cnl"].ptr, s["vxl"].ptr, s["vxl"].count,
                  ctypes.byref(found), s["ws"].ptr, s["ws"].nbytes, st)
        capi.call("raptr_sm_from_wq", su, g, s["cnl"].ptr, s["vxl"].ptr, s["val"].ptr,
                  found.value, nrays, seed, capi.RAYGEN_RAND, st)
        return [_tensor(s["cnl"]), _tensor(s["vxl"]), _tensor(s["val"])]
    if kind == "build":
        nnz = ctypes.c_int64()
        if case["count"]:
            capi.call("raptr_sm_build_csr_ex", su, g, s["d_list"].ptr, len(s["list"]), nrays,
                      seed, capi.RAYGEN_RAND, 0, s["row_ptr"].ptr, None, None, 0,
                      ctypes.byref(nnz), s["ws"].ptr, s["ws"].nbytes, st)
        capi.call("raptr_sm_build_csr_ex", su, g, s["d_list"].ptr, len(s["list"]), nrays, seed,
                  capi.RAYGEN_RAND, 0, s["row_ptr"].ptr, s["vxl"].ptr, s["val"].ptr,
                  nnz.value if case["count"] else s["vxl"].count, ctypes.byref(nnz),
                  s["ws"].ptr, s["ws"].nbytes, st)
        return [_tensor(s["row_ptr"]), _tensor(s["vxl"]), _tensor(s["val"])]
    if kind == "sens":
        return _tensor(sysmat.sensitivity(setup, grid, nrays, seed=seed, stream=st))
    if kind == "project":
        return [sysmat.forward_project(setup, grid, s["image"], nrays, s["list"], seed=seed),
                sysmat.backproject(setup, grid, nrays, s["list"], s["counts"], seed=seed)]
    if kind == "reco":
        A = sysmat.build_csr(setup, grid, s["list"], nrays, seed=seed, stream=st,
                             capacity="auto")
        R = Reconstructor(A, s["sens"], case["value_type"], 1, stream=st, row_order=setup)
        x = R.mlem(s["counts"], np.full(grid.nvox, 1.0 / grid.nvox, np.float32), case["niter"],
                   stream=st)
        R.close()
        return x
    x, x0 = s["x"], s["x0"]
    capi.call("raptr_memcpy_d2d", x.ptr, x0.ptr, x.nbytes, st)
    s["plan"].run(s["y"], x, case["niter"], case["frames"], stream=st)
    return _tensor(x, (grid.nvox, case["frames"]))


# ------------------------------------------------- what a pass must move
def _rows(case):
    """Measured rows of a case, about."""
    if "channels" in case:
        return case["channels"]
    allc = case["na"] * case["npix"] ** 4
    if case["kind"] == "sens":
        return allc
    return allc * (1.0 - math.exp(-case["events"] / (0.8 * allc)))


def _row_entries(case):
    """Non-zero voxels per matrix row, about: the path inside the grid in
    voxel steps times the cross-section of the 4 mm wide tube of rays."""
    n = (case["nx"] * case["ny"] * case["nz"]) ** (1.0 / 3.0)
    width = min(4.0 / case["pitch"] + 0.8, 0.9 * case["nrays"] ** 0.5)
    return n * width * width


def _pairs(case):
    """Voxels within the sum of the radii of a channel's line, about."""
    n = case["nx"] * case["ny"] * case["nz"]
    radius = 0.5 * (math.sqrt(3.0) * case["pitch"] + math.sqrt(4.0 ** 2 + 4.0 ** 2 + 20.0 ** 2))
    side = n ** (1.0 / 3.0) * case["pitch"]
    return n * min(1.0, math.pi * radius ** 2 / side ** 2)


def _capacity(case):
    """Entries of the buffers a program holds for a list of this length; the
    part past the last entry stays zero."""
    n = case["nx"] * case["ny"] * case["nz"]
    per = 1.5 * _pairs(case) if case["kind"] == "workqueue" else 2.5 * _row_entries(case) + 100
    return int(min(per, n) * case["channels"])


def work(case):
    kind, nr, n = case["kind"], case["nrays"], case["nx"] * case["ny"] * case["nz"]
    rows, per = _rows(case), _row_entries(case)
    nnz = rows * per
    # a ray's end points (twenty 32-bit multiplies each way and the
    # transformation), then a subtraction, a division and the slab
    # comparisons per crossed plane
    rays = rows * nr * (150.0 + 12.0 * (case["nx"] + case["ny"] + case["nz"]) / 3.0 * 2.0)
    if kind == "workqueue":
        pairs = rows * _pairs(case)
        return {"bytes": 4.0 * rows + 12.0 * pairs, "flops": 20.0 * pairs + rays}
    if kind == "build":
        return {"bytes": 12.0 * rows + 8.0 * nnz, "flops": rays}
    if kind == "sens":
        return {"bytes": 8.0 * n, "flops": rays + nnz}
    if kind == "project":
        return {"bytes": 2 * (4.0 + 8.0) * rows + 12.0 * n, "flops": 2 * (rays + 2.0 * nnz)}
    # an iteration streams the matrix once (value and 2-byte index): it is
    # larger than any cache at the sizes that matter
    frames, vb = case.get("frames", 1), {"f32": 4, "u16": 2, "f16": 2}[case["value_type"]]
    it = {"bytes": case["niter"] * ((vb + 2.0) * nnz + frames * (4.0 * rows + 12.0 * n)),
          "flops": case["niter"] * 4.0 * nnz * frames}
    if kind == "reco":
        it["bytes"] += 12.0 * rows + 8.0 * nnz
        it["flops"] += rays
    return it


# ------------------------------------------------------ the same in 64 bits
def _mulhilo(a, b):
    p = a * b  # a < 2^32 constant, b < 2^32: split so that int64 holds it
    lo = p & 0xFFFFFFFF
    hi = ((a * (b >> 16) + ((a * (b & 0xFFFF)) >> 16)) >> 16) & 0xFFFFFFFF
    return hi, lo


def _philox(c, k):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors."""
    c = list(c)
    k0, k1 = k
    for _ in range(10):
        h0, l0 = _mulhilo(0xD2511F53, c[0])
        h1, l1 = _mulhilo(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _angles(setup):
    """sin and cos of the C library's float functions per angle."""
    libm, f32 = ctypes.CDLL("libm.so.6"), np.float32
    out = []
    for f in (libm.sinf, libm.cosf):
        f.restype, f.argtypes = ctypes.c_float, [ctypes.c_float]
        out.append([f(f32(math.pi) * f32(k) * f32(setup.da) / f32(180)) for k in range(setup.na)])
    return torch.tensor(out, dtype=torch.float32, device="cuda")


def _rays(setup, channels, nrays, seed):
    """Single-precision ray ends [k, nrays, 6] of the channels: six uniforms
    of the counter (channel, ray, 0 | 1, 0) placed in the two pixels."""
    c = channels.to(torch.int64)
    rest, idx = c, []
    for n in (setup.n1y, setup.n1z, setup.n0y, setup.n0z):
        idx.append(rest % n)
        rest = rest // n
    sn, cs = (t[rest][:, None] for t in _angles(setup))
    cc = c[:, None].expand(-1, nrays)
    rr = torch.arange(nrays, device="cuda")[None].expand(len(c), -1)
    zero = torch.zeros_like(cc)
    w = (_philox([cc, rr, zero, zero], (seed & 0xFFFFFFFF, 0)) +
         _philox([cc, rr, zero + 1, zero], (seed & 0xFFFFFFFF, 0)))
    u = [((x >> 8) + 1).float() * (1.0 / 16777216.0) for x in w[:6]]
    f32 = np.float32
    e0, e1, e2 = (float(f32(v)) for v in (setup.segx, setup.segy, setup.segz))
    out = []
    for d, (pos, ny, nz) in enumerate(((setup.pos0x, setup.n0y, setup.n0z),
                                       (setup.pos1x, setup.n1y, setup.n1z))):
        iy, iz = (idx[2], idx[3]) if d == 0 else (idx[0], idx[1])
        p0 = float(f32(pos)) - 0.5 * e0
        p1 = (iy.float() - 0.5 * (ny - 1))[:, None] * e1
        p2 = (iz.float() - 0.5 * (nz - 1))[:, None] * e2 - 0.5 * e2
        b0, b1, b2 = u[3 * d:3 * d + 3]
        out += [cs * e0 * b0 + sn * e2 * b2 + (cs * p0 + sn * p2), e1 * b1 + (p1 - 0.5 * e1),
                -sn * e0 * b0 + cs * e2 * b2 + (-sn * p0 + cs * p2)]
    return torch.stack(out, 2)


def _pixel_centres(setup, channels):
    """The same transformation at the pixel centres, single precision."""
    c = channels.to(torch.int64)
    rest, idx = c, []
    for n in (setup.n1y, setup.n1z, setup.n0y, setup.n0z):
        idx.append(rest % n)
        rest = rest // n
    sn, cs = (t[rest] for t in _angles(setup))
    e0, e1, e2 = (float(np.float32(v)) for v in (setup.segx, setup.segy, setup.segz))
    out = []
    for pos, ny, nz, iy, iz in ((setup.pos0x, setup.n0y, setup.n0z, idx[2], idx[3]),
                                (setup.pos1x, setup.n1y, setup.n1z, idx[0], idx[1])):
        p0 = float(np.float32(pos)) - 0.5 * e0
        p1 = (iy.float() - 0.5 * (ny - 1)) * e1
        p2 = (iz.float() - 0.5 * (nz - 1)) * e2 - 0.5 * e2
        out.append(torch.stack([cs * e0 * 0.5 + sn * e2 * 0.5 + (cs * p0 + sn * p2),
                                e1 * 0.5 + (p1 - 0.5 * e1),
                                -sn * e0 * 0.5 + cs * e2 * 0.5 + (-sn * p0 + cs * p2)], 1))
    return out


def _div(a, b):
    """a / b, correctly rounded whatever the type."""
    return (a.double() / b.double()).to(a.dtype)


def _sqrt(a):
    return a.double().sqrt().to(a.dtype)


def _mean_chord(rays, row, box, dtype):
    """Mean over the rays of the slab intersection length of voxel boxes
    [k, 3, 2] with the rays of their rows."""
    a = torch.zeros(len(row), device="cuda", dtype=dtype)
    box = box.to(dtype)
    for r in range(rays.shape[1]):
        ray = rays[row, r].to(dtype)
        p, d = ray[:, :3], ray[:, 3:] - ray[:, :3]
        t = _div(box - p[:, :, None], d[:, :, None])
        lo, hi = t.amin(2), t.amax(2)
        lo = torch.where(d == 0, -math.inf, lo).amax(1)
        hi = torch.where(d == 0, math.inf, hi).amin(1)
        length = _sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2])
        a += torch.where(lo < hi, (hi - lo) * length, torch.zeros_like(lo))
    return a / rays.shape[1]


def _matrix64(setup, grid, nrays, seed, channels, pairs=1 << 22, values=True, drop=True):
    """Yields (rows, voxels, FP64 values) of the candidates near each
    channel's line; drop: those whose single-precision value is not zero."""
    n = torch.tensor(grid.n, device="cuda")
    o, d = (torch.tensor(v, dtype=torch.float32, device="cuda") for v in (grid.o, grid.d))
    v = torch.arange(grid.nvox, device="cuda")
    ijk = torch.stack([v // (grid.n[1] * grid.n[2]), v // grid.n[2] % grid.n[1], v % grid.n[2]], 1)
    centre = o + (ijk.float() + 0.5) * d
    radii = 0.5 * (np.float32(np.sqrt(sum(np.float32(x) ** 2 for x in grid.d))) +
                   np.float32(np.sqrt(sum(np.float32(x) ** 2 for x in
                                          (setup.segx, setup.segy, setup.segz)))))
    step = max(1, min(len(channels), 16 * pairs // grid.nvox))
    for first in range(0, len(channels), step):
        ch = channels[first:first + step]
        p0, p1 = _pixel_centres(setup, ch)
        ab = p1 - p0
        norm = _sqrt(ab[:, 0] * ab[:, 0] + ab[:, 1] * ab[:, 1] + ab[:, 2] * ab[:, 2])
        ap = [centre[None, :, k] - p0[:, None, k] for k in range(3)]
        ab = [ab[:, None, k] for k in range(3)]
        x = ab[1] * ap[2] - ab[2] * ap[1]
        s = x * x
        x = ab[2] * ap[0] - ab[0] * ap[2]
        s += x * x
        x = ab[0] * ap[1] - ab[1] * ap[0]
        s += x * x
        row, vox = (_div(_sqrt(s), norm[:, None]) < float(radii)).nonzero(as_tuple=True)
        del s, x, ap, ab
        rays = _rays(setup, ch, nrays, seed)
        for k in range(0, len(row), pairs):
            rw, vx = row[k:k + pairs], vox[k:k + pairs]
            if drop:
                box = torch.stack([o + ijk[vx].float() * d, o + (ijk[vx] + 1).float() * d], 2)
                keep = _mean_chord(rays, rw, box, torch.float32) != 0
                rw, vx = rw[keep], vx[keep]
            box = torch.stack([o + ijk[vx].float() * d, o + (ijk[vx] + 1).float() * d], 2)
            yield first + rw, vx, (_mean_chord(rays, rw, box, torch.float64) if values else None)


def _mlem64(m, n, row, col, val, y, sens, niter):
    """The recurrence in FP64 on a matrix given as row-sorted entries."""
    y = y.double().reshape(m, -1)
    rp = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.bincount(row, minlength=m).cumsum(0)
    A = torch.sparse_csr_tensor(rp.int(), col.int(), val.double(), (m, n))
    by_col = col.sort(stable=True).indices
    cp = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    cp[1:] = torch.bincount(col, minlength=n).cumsum(0)
    At = torch.sparse_csr_tensor(cp.int(), row[by_col].int(), val[by_col].double(), (n, m))
    del by_col, row, col
    s = torch.as_tensor(sens, device="cuda")
    s = (s / s.sum())[:, None]
    s = s + (s == 0)
    x = torch.full((n, y.shape[1]), 1.0 / n, dtype=torch.float64, device="cuda")
    for _ in range(niter):
        yt = A @ x
        e = torch.where((yt != 0) & (y != 0), y / yt, torch.zeros_like(y))
        x = x * (At @ e) / s
        x = x / x.sum(0)
    return x


def exact(case, seed):
    setup, grid, kind, nrays = _setup(case), _grid(case), case["kind"], case["nrays"]
    s = int(seed) & 0x7fffffff
    rows = _rows(case)
    # slab tests of the candidates, about 1e11 in ten seconds
    tests = rows * nrays * min(grid.nvox, 60.0 * (grid.nvox ** (1 / 3)) * (4.0 / case["pitch"] ** 2))
    if kind != "recon" and tests > 5e10:
        return None
    if kind in ("workqueue", "build", "project"):
        lst, y = _list(case, setup, grid, seed)
        got = list(_matrix64(setup, grid, nrays, s, lst, drop=kind != "workqueue"))
        row, vox, val = (torch.cat(t) for t in zip(*got))
        if kind != "project":
            full = torch.zeros(_capacity(case), dtype=torch.float64, device="cuda")
            full[:len(val)] = val
            return [None, None, full]
        image = torch.rand(grid.nvox, generator=_generator(seed, 4), device="cuda").double()
        out = torch.zeros(len(lst), dtype=torch.float64, device="cuda")
        back = torch.zeros(grid.nvox, dtype=torch.float64, device="cuda")
        out.index_add_(0, row, val * image[vox])
        back.index_add_(0, vox, val * y[row].double())
        return [out, back / back.sum()]
    if kind == "sens":
        out = torch.zeros(grid.nvox, dtype=torch.float64, device="cuda")
        for _, vox, val in _matrix64(setup, grid, nrays, s,
                                     torch.arange(setup.nchannels, device="cuda")):
            out.index_add_(0, vox, val)
        return out
    meas, y = _counts(case, setup, grid, seed)
    sens = _sensitivity(case, setup, grid)
    if kind == "reco":
        got = list(_matrix64(setup, grid, nrays, s, meas))
        row, col, val = (torch.cat(t) for t in zip(*got))
        return _mlem64(len(meas), grid.nvox, row, col, val, y, sens, case["niter"]).flatten()
    # the matrix is this case's input
    A = sysmat.build_csr(setup, grid, meas.cpu().numpy(), nrays, seed=1, capacity="auto")
    rp = _tensor(A.row_ptr, (A.m + 1,))
    row = torch.repeat_interleave(torch.arange(A.m, device="cuda"), rp[1:] - rp[:-1])
    return _mlem64(A.m, grid.nvox, row, _tensor(A.col, (A.nnz,)).long(),
                   _tensor(A.val, (A.nnz,)), y, sens, case["niter"])
