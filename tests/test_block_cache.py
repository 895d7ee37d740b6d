"""The cache of freed device blocks: its rules over a model of the driver
(tests/cpp/test_block_cache.cpp) and its entry points on the device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "raptr_amd", "lib", "test_block_cache")


def test_rules_over_a_model_driver():
    if not os.path.exists(EXE):
        pytest.fail(f"{EXE} not built (run __graft_entry__.build())")
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "0 failure(s)" in r.stdout, r.stdout + r.stderr


@pytest.mark.gpu
def test_free_twice_is_refused(gpu):
    """A second raptr_free of a block is an error, and the block is handed out
    once."""
    import ctypes as C
    from raptr_amd import _capi as capi
    L = capi.lib()
    nb = 9 << 20
    p, q, r = C.c_void_p(), C.c_void_p(), C.c_void_p()
    capi.call("raptr_malloc", C.byref(p), nb)
    capi.call("raptr_free", p)
    assert L.raptr_free(p) == capi.RAPTR_ERR_DEVICE
    capi.call("raptr_malloc", C.byref(q), nb)
    capi.call("raptr_malloc", C.byref(r), nb)
    assert q.value != r.value
    capi.call("raptr_free", q)
    capi.call("raptr_free", r)


@pytest.mark.gpu
def test_handed_out_blocks_are_cleared(gpu):
    import numpy as np
    from raptr_amd.device import DeviceArray
    for n in (3 << 20, 17 << 20):
        for _ in range(3):
            a = DeviceArray(n, np.uint8)
            assert not a.numpy().any()
            a.copy_from(np.full(n, 0xA5, np.uint8))
            a.free()


def _capture(stream, work, beside):
    """work() captured on the stream in thread-local mode while beside() runs
    in another thread; the capture's end status and the graph's nodes."""
    import ctypes as C
    import threading
    H = C.CDLL("libamdhip64.so")
    vp = C.c_void_p
    failed = []

    def run():
        try:
            beside()
        except Exception as e:  # noqa: BLE001 - reported by the caller's assert
            failed.append(e)
    graph = vp()
    assert H.hipStreamBeginCapture(vp(stream.handle), 1) == 0
    work()
    t = threading.Thread(target=run)
    t.start()
    t.join()
    work()
    status = H.hipStreamEndCapture(vp(stream.handle), C.byref(graph))
    n = C.c_size_t()
    if graph.value:
        assert H.hipGraphGetNodes(graph, None, C.byref(n)) == 0
        assert H.hipGraphDestroy(graph) == 0
    assert not failed, failed
    return status, n.value


@pytest.mark.gpu
def test_frees_leave_a_capture_of_another_thread(gpu):
    """Blocks, and a plan with its blocks, freed while another thread captures:
    the capture ends well and holds all of its work."""
    import numpy as np
    from raptr_amd import sysmat
    from raptr_amd.device import DeviceArray, Stream
    from raptr_amd.geometry import config_tiny
    from raptr_amd.recon import Reconstructor
    setup, grid, nrays = config_tiny()
    A = sysmat.build_csr(setup, grid, np.arange(setup.nchannels, dtype=np.int32), nrays)
    sens = sysmat.sensitivity(setup, grid, nrays)
    R = Reconstructor(A, sens, "f32", 1, row_order=setup)
    dy = DeviceArray.from_numpy(np.ones(A.m, np.float32))
    dx = DeviceArray.from_numpy(np.full(A.n, 1.0 / A.n, np.float32))
    st = Stream()

    def work():
        R.run(dy, dx, 1, use_graph=False, stream=st.handle)
    blocks = [DeviceArray(n, np.uint8) for n in (1 << 12, 9 << 20, 64 << 20)]
    plans = [Reconstructor(A, sens, "f32", 1, row_order=setup) for _ in range(2)]
    other = Stream()
    dz = DeviceArray.from_numpy(np.full(A.n, 1.0 / A.n, np.float32))
    plans[0].run(dy, dz, 5, stream=other.handle)  # a plan with captured iterations
    other.sync()

    def frees():
        for b in blocks:
            b.free()
        for p in plans:
            p.close()
        DeviceArray(9 << 20, np.uint8).free()  # a kept block, handed out and freed
    status, alone = _capture(st, work, lambda: None)
    assert status == 0 and alone >= 2
    assert _capture(st, work, frees) == (0, alone)


@pytest.mark.gpu
def test_cached_blocks_go_back_on_request(gpu):
    """Free memory as the driver counts it: a freed block returns to it with
    release_cached; mem_info counts it throughout."""
    import ctypes as C
    import numpy as np
    from raptr_amd.device import DeviceArray, mem_info, release_cached
    H = C.CDLL("libamdhip64.so")
    f, t = C.c_size_t(), C.c_size_t()

    def driver_free():
        assert H.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value
    # (the driver's count also moves by chunks of its own: blocks, half of one)
    nb, half = 512 << 20, 256 << 20
    release_cached()
    before = driver_free()
    a = DeviceArray(nb, np.uint8)
    assert driver_free() <= before - half
    held = mem_info()[0]
    a.free()
    assert driver_free() <= before - half
    assert mem_info()[0] >= held + half
    release_cached()
    assert driver_free() >= before - half


@pytest.mark.gpu
def test_threads_build_run_and_free_plans(gpu):
    """Four threads with plans and streams of their own, buffers new for every
    run: each run captures while others allocate and free."""
    import threading
    import numpy as np
    from raptr_amd import sysmat
    from raptr_amd.device import DeviceArray, Stream
    from raptr_amd.geometry import config_small
    from raptr_amd.recon import Reconstructor
    setup, grid, nrays = config_small()
    A = sysmat.build_csr(setup, grid, np.arange(8000, dtype=np.int32), nrays)
    sens = sysmat.sensitivity(setup, grid, nrays)
    y = np.random.default_rng(0).poisson(5, A.m).astype(np.float32)
    x0 = np.full(A.n, 1.0 / A.n, np.float32)
    want = Reconstructor(A, sens, "f32", 1, row_order=setup).mlem(y, x0, 9)
    wrong = []

    def work(t):
        try:
            st = Stream()
            for k in range(10):
                R = Reconstructor(A, sens, "f32", 1, row_order=setup, stream=st.handle)
                for _ in range(2):
                    if not np.array_equal(R.mlem(y, x0, 9, stream=st.handle), want):
                        wrong.append((t, k))
                DeviceArray(5000000 + 100000 * k, np.uint8).free()
                R.close()
        except Exception as e:  # noqa: BLE001 - reported below
            wrong.append((t, repr(e)))
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
