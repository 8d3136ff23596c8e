"""Float32 products in pipelined tiles whose reads and transfers lie among the products: as few stages of 32 k as there can be (fewer than the
ring holds), rows and columns around the edges of tiles, rows apart by more than K, and the widths from which few rows take them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n,k", [
    (65, 130, 32), (65, 300, 64), (97, 129, 96), (129, 128, 128), (200, 4100, 32), (1000, 8200, 96),  # one to four stages
    (17, 14208, 64), (17, 14209, 64), (32, 14340, 544), (24, 33000, 96),                              # 17 to 32 rows: 111 tiles and more
    (33, 8064, 64), (33, 8065, 64), (64, 8196, 544), (40, 33000, 288),                                # 33 to 64 rows: 63 tiles and more
])
def test_products_in_tiles_match_64_bit_sums_and_single_rows(rows, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(rows + n + k)
    # rows apart by 12 more than K, and not-a-numbers around everything that is to be read
    x = torch.full((rows + 1, k + 12), float("nan"), device="cuda")
    w = torch.full((n + 1, k + 12), float("nan"), device="cuda")
    x[:rows, :k] = torch.randn(rows, k, generator=gen).cuda()
    w[:n, :k] = torch.randn(n, k, generator=gen).cuda()
    x, w = x[:rows, :k], w[:n, :k]
    out = torch.full((rows, n), float("nan"), device="cuda")
    kn.linear(x, w, out)
    want = x.double() @ w.double().T
    # chunks of 256 k in one chain each, then the chunks: at most 256 + k / 256 roundings of 2^-24 of sum |x| |w|
    assert ((out - want).abs() <= (256 + k / 256) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()
    one = torch.empty(1, n, device="cuda")
    for r in (0, rows // 2, rows - 1):
        kn.linear(x[r : r + 1], w, one)
        assert torch.equal(out[r : r + 1], one), r


@pytest.mark.parametrize("rows,n,k", [(65, 65, 32), (90, 4100, 96), (70, 16600, 288), (129, 32768, 64), (40, 33000, 64)])
@pytest.mark.parametrize("which", ["x", "w"])
def test_rows_beyond_32_bit_offsets(rows, n, k, which):
    """A tile's rows 2^31 bytes apart from first to last: the bits of the same rows side by side."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, apart = HipKernels(), 2 ** 22
    n = min(n, 300) if which == "w" else n
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda") for r in (rows, n))
    near = x if which == "x" else w
    far = torch.empty((len(near) - 1) * apart + k, device="cuda").as_strided(near.shape, (apart, 1))
    far.copy_(near)
    want, out = torch.empty(rows, n, device="cuda"), torch.full((rows, n), float("nan"), device="cuda")
    kn.linear(x, w, want)
    kn.linear(*((far, w) if which == "x" else (x, far)), out)
    assert torch.equal(out, want)
