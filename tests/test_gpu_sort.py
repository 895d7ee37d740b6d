"""The radix sort around its tiles (2,048 pairs in sorts of up to 2^20, 4,096 in
longer ones), through raptr_coo_sort, against numpy's stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 4097, 100003, (1 << 20) - 1, 1 << 20,
                               (1 << 20) + 1, (1 << 20) + 4096, 2500001])
@pytest.mark.parametrize("keys", ["few", "many"])
def test_coo_sort_tiles(gpu, n, keys):
    from raptr_amd import sparse
    rng = np.random.default_rng(n)
    top = 3 if keys == "few" else 70000
    row = rng.integers(0, top, n).astype(np.int32)
    col = rng.integers(0, top, n).astype(np.int32)
    val = rng.random(n).astype(np.float32)
    order = np.lexsort((col, row))
    got = sparse.coo_sort(val, row, col)
    np.testing.assert_array_equal(got[1], row[order])
    np.testing.assert_array_equal(got[2], col[order])
    np.testing.assert_array_equal(got[0], val[order])  # equal keys keep their order
