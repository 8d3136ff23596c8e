"""Products of at most 8 rows and 8 columns a compute unit, around the edges of chunks of 128 k and blocks of 8 columns."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 5, 7, 8])
@pytest.mark.parametrize("n,k", [(1, 512), (8, 640), (9, 2048), (136, 2176), (1000, 4096), (1536, 5376), (2048, 512), (2048, 1920), (2048, 8320)])
def test_products(rows, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(n + k)
    x, w = torch.randn(rows, k + 8, generator=gen).bfloat16().cuda()[:, :k], torch.randn(n, k, generator=gen).bfloat16().cuda()
    want = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)  # (products of bfloat16 are exact; a rounding a term)
    wide = torch.full((rows, n + 5), 7.0, device="cuda")
    for held in (w, kn.pack_weight(w)):
        kn.linear(x, held, wide[:, :n])
        assert ((wide[:, :n] - want).abs() <= bound).all() and bool((wide[:, n:] == 7.0).all())
    narrow = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
    kn.linear(x, w, narrow)
    assert ((narrow - want).abs() <= bound + 2.0 ** -8 * want.abs()).all()
    # an infinity or NaN in one row or column stays there
    x2, w2 = x.clone(), w.clone()
    x2[0, k - 1], w2[n - 1, 3] = float("inf"), float("nan")
    kn.linear(x2, w2, wide[:, :n])
    assert not bool(wide[0, :n].isfinite().any()) and bool(wide[:, n - 1].isnan().all())
    if rows > 1 and n > 1:
        assert ((wide[1:, : n - 1] - want[1:, : n - 1]).abs() <= bound[1:, : n - 1]).all()


@pytest.mark.parametrize("rows,k", [(1, 512), (4, 8192), (8, 4096), (8, 8192), (3, 2176)])
def test_into_the_stream(rows, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, n = HipKernels(), 2048
    gen = torch.Generator().manual_seed(k)
    act, w = torch.randn(rows, k, generator=gen).bfloat16().cuda(), kn.pack_weight(torch.randn(n, k, generator=gen).bfloat16().cuda() * 0.1)
    x, gain = torch.randn(rows, n, generator=gen).cuda(), torch.randn(n, generator=gen).cuda()
    plain = torch.empty(rows, n, device="cuda")
    kn.linear(act, w, plain)
    parts = kn.linear_fused_parts(torch.bfloat16, rows, n, k)
    assert parts > 0
    sq, scaled, got = torch.full((rows, parts), 7.0, device="cuda"), torch.empty(rows, n, dtype=torch.bfloat16, device="cuda"), x.clone()
    kn.linear_residual(act, w, got, sq, gain=gain, scaled=scaled)
    assert torch.equal(got, x + plain) and torch.equal(scaled, (got * gain).bfloat16())
    assert ((sq.double().sum(1) - (got.double() ** 2).sum(1)).abs() <= 2048 * 2.0 ** -24 * (got.double() ** 2).sum(1)).all()


@pytest.mark.parametrize("n,k", [(320, 4096), (1000, 4096), (1536, 5376), (2040, 2176), (2040, 2048), (2040, 8320)])
@pytest.mark.parametrize("rows", [1, 3, 8])
def test_streamed_products_sum_in_the_same_order(rows, n, k):
    """The same columns, of a weight whose columns are not in eights, which goes in pairs of chunks, and of one that may be streamed."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda").bfloat16() for r in (rows, n + 1))
    want, got = torch.empty(rows, n + 1, device="cuda"), torch.empty(rows, n, device="cuda")
    kn.linear(x, w, want)
    kn.linear(x, w[:n], got)
    assert torch.equal(got, want[:, :n])


def squares_of_eights(x):
    """Sums of the squares of 8 neighbours in the order of both kernels: those of columns 4 apart with one rounding, then sums."""
    v = x.reshape(len(x), -1, 8)
    # (a product of two 24-bit numbers and a third number, exact in 64 bits but for the rarest of sums, rounded once)
    first = (v[..., :4].double() ** 2 + (v[..., 4:] ** 2).double()).float()
    return (first[..., 0] + first[..., 2]) + (first[..., 1] + first[..., 3])


@pytest.mark.parametrize("rows,k", [(1, 2048), (2, 8192), (4, 512), (4, 8192), (3, 14464), (8, 1920), (8, 2048), (8, 4096)])
def test_streamed_products_of_2048_columns_sum_in_the_same_order(rows, k):
    """Every way out of a product of 8 columns a compute unit."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, n = HipKernels(), 2048
    gen = torch.Generator(device="cuda").manual_seed(k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda").bfloat16() for r in (rows, n))
    old = torch.randn(rows, n, generator=gen, device="cuda")
    want = torch.empty(rows, n, device="cuda")
    kn.linear(x, w[: n - 1], want[:, : n - 1])
    kn.linear(x, w[1:], want[:, 1:])
    acted = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
    kn.activation(want, acted, "relu2")
    for held in (w, kn.pack_weight(w)):
        wide, narrow, unit = torch.empty_like(want), torch.empty_like(acted), torch.empty_like(acted)
        kn.linear(x, held, wide)
        kn.linear(x, held, narrow)
        kn.linear_unit(x, held, unit, "relu2")
        new, sq = old.clone(), torch.empty(rows, kn.linear_fused_parts(torch.bfloat16, rows, n, k), device="cuda")
        kn.linear_residual(x, held, new, sq)
        parts = squares_of_eights(new)
        assert torch.equal(sq, parts)
        assert torch.equal(wide, want) and torch.equal(narrow, want.bfloat16()) and torch.equal(unit, acted) and torch.equal(new, old + want)


@pytest.mark.parametrize("rows,n,k,whole", [(1, 128, 2048, True), (8, 64, 4096, True), (8, 288, 8192, False), (9, 128, 2048, False),
                                            (3, 160, 2112, False), (2, 4096, 4096, False)])
def test_whole_or_in_pieces_added_up(rows, n, k, whole):
    from types import SimpleNamespace

    from longbow_quarrel_amd.kernels.hip import HipKernels
    from longbow_quarrel_amd.parts.base import project_narrow

    kn = HipKernels()
    assert kn.linear_whole(torch.bfloat16, rows, n, k) == whole and not kn.linear_whole(torch.float32, rows, n, k)
    gen = torch.Generator().manual_seed(n + k)
    x, w = torch.randn(rows, k, generator=gen).bfloat16().cuda(), torch.randn(n, k, generator=gen).bfloat16().cuda()
    out = torch.empty(rows, n, device="cuda")
    ws = SimpleNamespace(alloc=lambda shape, dtype, **_: torch.empty(shape, dtype=dtype, device="cuda"))
    project_narrow(kn, SimpleNamespace(ws=ws, kernels=kn), x, w, out)
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((out - x.double() @ w.double().T).abs() <= bound).all()
