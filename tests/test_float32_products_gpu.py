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


@pytest.mark.parametrize("n,k", [(4104, 4384), (8200, 2336), (6150, 6176), (4112, 2048), (4112, 2080),  # 8 wavefronts
                                 (4096, 4384), (2064, 8224), (4096, 4128), (1000, 12288)])              # 16
def test_streamed_rows_over_several_rounds_of_chunks(n, k):
    """At most 16 rows whose wavefronts take more than one chunk of 256 k each, with a part chunk or none at the end: the bits of
    pipelined tiles, and not-a-numbers around the operands and in a row and a column that stay there."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x, w = (torch.full((r + 1, k + 32), float("nan"), device="cuda") for r in (80, n))
    x[:80, :k], w[:n, :k] = (torch.randn(r, k, generator=gen, device="cuda") for r in (80, n))
    x, w = x[:80, :k], w[:n, :k]
    want = torch.empty(80, n, device="cuda")
    kn.linear(x, w, want)  # (tiles)
    exact, terms = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # chunks of 256 k in one chain each, then the chunks: at most 256 + k / 256 roundings of 2^-24 of sum |x| |w|
    assert ((want - exact).abs() <= (256 + k / 256) * 2.0 ** -24 * terms).all()
    for rows in (1, 4, 16):
        out = torch.full((rows + 1, n + 3), 7.0, device="cuda")
        kn.linear(x[:rows], w, out[:rows, :n])
        assert torch.equal(out[:rows, :n], want[:rows]), rows
        assert bool((out[rows] == 7).all()) and bool((out[:, n:] == 7).all())
    w[n - 1, k - 1], x[3, 0] = float("nan"), float("inf")
    out = torch.empty(16, n, device="cuda")
    kn.linear(x[:16], w, out)
    assert bool(out[:, n - 1].isnan().all()) and not bool(out[3].isfinite().any())
    clean = [r for r in range(16) if r != 3]
    assert torch.equal(out[clean, : n - 1], want[clean, : n - 1])


@pytest.mark.parametrize("n", [2048, 6144])
def test_a_row_has_the_same_bits_in_every_tile_of_a_wide_weight(n):
    """Numbers of rows around the edges of tiles of 32, 64, 96 and 128, each of which some of these launches take."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, k = HipKernels(), 544
    gen = torch.Generator().manual_seed(n)
    x, w = torch.randn(1201, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    some = [0, 1, 31, 32, 63, 64, 95, 96, 97, 127, 128, 129, 191, 288, 330, 575, 863, 1151, 1152, 1199, 1200]
    one = torch.empty(1201, n, device="cuda")
    for r in some:
        kn.linear(x[r : r + 1], w, one[r : r + 1])
    for rows in (65, 95, 96, 97, 161, 257, 289, 333, 600, 865, 1000, 1153, 1201):
        out = torch.full((rows, n), float("nan"), device="cuda")
        kn.linear(x[:rows], w, out)
        mine = [r for r in some if r < rows]
        assert torch.equal(out[mine], one[mine]), rows
        assert bool(out.isfinite().all()), rows
