"""Single tokens of a float32 run: four wavefronts a row and head (head sizes in 64s) make the bits of a prompt's last row, at lengths
around the ends of chunks of 64 keys, of 16 keys and of windows."""
import pytest
import torch

from test_kernels_gpu import kn, rel_err, run_attention  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(4, 2, 64), (2, 1, 128), (3, 3, 192), (2, 1, 256)])
@pytest.mark.parametrize("window", [0, 70])
def test_single_tokens(kn, heads, kv_heads, head_dim, window):  # noqa: F811
    lengths = [1, 15, 16, 63, 64, 65, 130, 193]
    whole, want = run_attention(kn, None, lengths, lengths, heads, kv_heads, head_dim, torch.float32, 5, window=window,
                                force_generic=True, q_by_position=True)
    assert rel_err(whole, want) < 2e-6
    single, _ = run_attention(kn, None, lengths, [1] * len(lengths), heads, kv_heads, head_dim, torch.float32, 5, window=window,
                              decode=True, force_generic=True, q_by_position=True)
    for b in range(len(lengths)):
        assert torch.equal(single[b], whole[sum(lengths[: b + 1]) - 1]), b


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(4, 1, 64), (8, 2, 128), (8, 1, 192), (4, 1, 256), (6, 1, 128), (10, 5, 64), (2, 1, 192)])
@pytest.mark.parametrize("window", [0, 70])
def test_heads_of_a_group_together(kn, heads, kv_heads, head_dim, window):  # noqa: F811
    """Groups of 8, 6, 4 and 2 heads, four or two of which a workgroup takes together: the bits of a prompt's last row."""
    lengths = [1, 16, 64, 65, 193]
    whole, want = run_attention(kn, None, lengths, lengths, heads, kv_heads, head_dim, torch.float32, 6, window=window,
                                force_generic=True, q_by_position=True)
    assert rel_err(whole, want) < 2e-6
    single, _ = run_attention(kn, None, lengths, [1] * len(lengths), heads, kv_heads, head_dim, torch.float32, 6, window=window,
                              decode=True, force_generic=True, q_by_position=True)
    for b in range(len(lengths)):
        assert torch.equal(single[b], whole[sum(lengths[: b + 1]) - 1]), b
