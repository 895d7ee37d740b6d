"""Plans whose (row block, column) keys need more than 32 bits: 33,000 blocks of
one row and 65,536 columns, so 2^31 segments and more, against the same matrix
in default blocks and against the FP64 recurrence."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M, N = 33000, 65536


@pytest.fixture(scope="module")
def system(gpu):
    from raptr_amd.device import DeviceArray
    from raptr_amd.sysmat import DeviceCSR
    rng = np.random.default_rng(1)
    # columns of the first, the last and some rows at both ends of the range
    col = np.sort(rng.integers(0, 2000, (M, 3)) * 32 + rng.integers(0, 10, (M, 3)), axis=1)
    col += np.arange(3) * 11  # distinct
    col[::97, 2] = N - 1
    col[::89, 0] = 0
    col[-1] = (0, 40000, N - 1)
    assert (np.diff(col, axis=1) > 0).all()
    row = np.repeat(np.arange(M), 3)
    col = col.reshape(-1).astype(np.int32)
    val = rng.uniform(0.5, 2.0, len(col)).astype(np.float32)
    A = DeviceCSR(M, N, len(col), DeviceArray.from_numpy(np.arange(M + 1, dtype=np.int64) * 3),
                  DeviceArray.from_numpy(col), DeviceArray.from_numpy(val))
    sens = np.bincount(col, val.astype(np.float64), N)
    y = rng.integers(0, 9, M).astype(np.float32)
    x = np.full(N, 1.0 / N)
    s = sens / sens.sum()
    s = s + (s == 0)
    for _ in range(3):
        yt = np.bincount(row, val * x[col], M)
        e = np.divide(y, yt, out=np.zeros(M), where=yt != 0)
        x = x * np.bincount(col, val * e[row], N) / s
        x /= x.sum()
    return A, DeviceArray.from_numpy(sens), y, x


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def test_keys_of_33_bits_single_frame(system):
    """1e-5 against FP64 (FP32 sums of three terms a row and a few a column),
    1e-6 against the same sums in other blocks."""
    from raptr_amd.recon import Reconstructor
    A, sens, y, want = system
    x0 = np.full(N, 1.0 / N, np.float32)
    base = Reconstructor(A, sens, "f32", 1)
    a = base.mlem(y, x0, 3)
    base.close()
    R = Reconstructor(A, sens, "f32", 1, block_rows=1)
    assert R.info()["row_blocks"] == M
    R.set_fused(False)  # the row-blocked transpose
    x = R.mlem(y, x0, 3)
    R.close()
    assert _rel(x, want) <= 1e-5 and _rel(x, a) <= 1e-6


def test_keys_of_33_bits_64_frames(system):
    from raptr_amd.recon import Reconstructor
    A, sens, y, want = system
    Y = np.repeat(y[:, None], 64, axis=1)
    Y[:, 1:32] *= 2.0
    R = Reconstructor(A, sens, "f32", 64, block_rows=1, grouped_only=True)
    X = R.mlem(Y, np.full((N, 64), 1.0 / N, np.float32), 3)
    R.close()
    for f in (0, 1, 63):  # a count scale leaves the normalised image alone
        assert _rel(X[:, f], want) <= 1e-5
