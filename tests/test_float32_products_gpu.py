"""True 32-bit products: a row has the same bits alone as in every launch, whichever kernel and tile takes it (up to 16, 32
and 64 rows with 8 or 16 wavefronts, pipelined tiles of 64 and 128 rows, the size-agnostic tiles)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(272, 2336), (4112, 544), (16500, 512), (130, 36), (200, 2080)])
def test_a_row_has_the_same_bits_in_every_launch(n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(n + k)
    x, w = torch.randn(300, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    one = torch.empty(300, n, device="cuda")
    for r in range(300):
        kn.linear(x[r : r + 1], w, one[r : r + 1])
    want = x.double() @ w.double().T
    # chunks of 256 k in one chain each, then the chunks: at most 256 + k / 256 roundings of 2^-24 of sum |x| |w|
    assert ((one - want).abs() <= (256 + k / 256) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()
    for rows in (2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 193, 300):
        out = torch.full((rows, n), float("nan"), device="cuda")
        kn.linear(x[:rows], w, out)
        assert torch.equal(out, one[:rows]), rows
