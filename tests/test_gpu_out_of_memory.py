"""A plan whose union counts find no device memory: RAPTR_ERR_OUT_OF_MEMORY, not
a device error, and the next plan is whole.  Runs in a process of its own, with
a hipMalloc that fails for blocks of one size."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "raptr_amd", "lib", "failing_malloc.so")

CODE = """
import ctypes as C, sys
F = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
import numpy as np
from raptr_amd import _capi as capi, sysmat
from raptr_amd.geometry import config_small
from raptr_amd.recon import Reconstructor
setup, grid, nrays = config_small()
rows = 17000
A = sysmat.build_csr(setup, grid, np.arange(rows, dtype=np.int32), nrays)
sens = sysmat.sensitivity(setup, grid, nrays)
Reconstructor(A, sens, "f32", 1).close()
fail, failed = C.c_size_t.in_dll(F, "fail_bytes"), C.c_int.in_dll(F, "failed")
fail.value = 8 * ((rows + 15) // 16)  # the only size of at least 1,024 groups
try:
    Reconstructor(A, sens, "f32", 1)
    status = capi.RAPTR_OK
except capi.RaptrError as e:
    status = e.status
n, fail.value = failed.value, 0
R = Reconstructor(A, sens, "f32", 1)
assert R.unions()["rows"] == 16
R.close()
print("failed", n, "status", status, "expected", capi.RAPTR_ERR_OUT_OF_MEMORY)
sys.exit(0 if n >= 1 and status == capi.RAPTR_ERR_OUT_OF_MEMORY else 1)
"""


@pytest.mark.gpu
def test_union_counts_without_memory(gpu):
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} not built (run __graft_entry__.build())")
    r = subprocess.run([sys.executable, "-c", CODE.format(lib=LIB)], capture_output=True,
                       text=True, timeout=100, cwd=ROOT)
    assert r.returncode == 0, r.stdout + r.stderr
