"""Which way products go, asked of the library's host functions (they run anywhere, as for 256 compute units)."""
import ctypes

import pytest

from longbow_quarrel_amd import build

F32, BF16 = 0, 1


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(build.ensure_built())


def test_a_few_rows_of_a_narrow_weight_and_a_short_k_are_not_shared_out(lib):
    for m in (17, 24, 32):
        for n in (128, 1024, 1536):
            assert [lib.lq_linear_splits(BF16, m, n, k, 0) for k in (512, 576, 960)] == [1, 1, 1]
            assert min(lib.lq_linear_splits(BF16, m, n, k, 0) for k in (1024, 2048, 4096)) > 1
    assert lib.lq_linear_splits(BF16, 33, 1024, 512, 0) == 2
