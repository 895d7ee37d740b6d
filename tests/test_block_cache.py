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
