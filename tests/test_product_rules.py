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


@pytest.mark.parametrize("heads,dk,dv,lengths,chunks", [
    # microseconds measured, token by token and in chunks
    (16, 64, 128, [300], True),                # 99, 37
    (16, 64, 128, [300] + [1] * 128, False),   # 160, 405
    (16, 64, 128, [48] + [1] * 128, False),    # 77, 387
    (16, 64, 128, [64] * 96, False),           # 261, 357
    (16, 128, 256, [64] + [1] * 128, False),   # 554, 740
    (16, 128, 256, [300] + [1] * 16, True),    # 236, 117
    (8, 128, 256, [512] + [1] * 64, True),     # 381, 193
    (4, 64, 64, [200] * 96, False),            # 109, 195
    (8, 32, 64, [512] + [1] * 64, False),      # 53 (in segments), 92
    (8, 128, 256, [3000], True)])
def test_gated_linear_attention_goes_in_chunks_where_that_is_faster(lib, heads, dk, dv, lengths, chunks):
    assert lib.lq_gla_scan_in_chunks(sum(lengths), len(lengths), heads, dk, dv, max(lengths)) == chunks


@pytest.mark.parametrize("heads,dk,dv,lengths,channel,chunks", [
    # microseconds measured, token by token and in chunks
    (16, 64, 64, [200] + [1] * 16, 0, True),     # 73, 49
    (16, 128, 128, [200] + [8] * 16, 0, True),   # 93, 70
    (8, 64, 128, [200] + [1] * 70, 0, True),     # 80, 59
    (16, 128, 128, [64], 0, False),              # 30, 32
    (16, 64, 64, [130] * 8, 1, False),           # 64, 78
    (16, 64, 64, [512] * 16, 1, False),          # 261, 368
    (32, 128, 128, [64] + [1] * 70, 1, False),   # 329, 384
    (16, 128, 128, [2048], 0, True)])            # 654, 146
def test_the_delta_rule_goes_in_chunks_where_that_is_faster(lib, heads, dk, dv, lengths, channel, chunks):
    assert lib.lq_delta_scan_in_chunks(sum(lengths), len(lengths), heads, dk, dv, max(lengths), channel) == chunks


def test_what_gated_linear_attention_does_not_take_in_chunks(lib):
    for sizes in ((0, 1, 8, 128, 256, 0), (500, 1, 8, 129, 256, 500), (47, 1, 8, 128, 256, 47), (3000, 1, 0, 128, 256, 3000)):
        assert lib.lq_gla_scan_in_chunks(*sizes) == 0
