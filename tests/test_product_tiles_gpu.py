"""Products of 17 rows and more: every tile that the estimate of a product's time can name, at its edges, whole and in shares of
K, tiles that are no multiple of the eight XCDs, columns left over from whole rounds of tiles, and groups of rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def within(got, x, w, rounded=0.0):
    """A sum of K products of bfloat16 (exact in 32 bits): at most K roundings of 2^-24 of the terms' absolute sum, in any
    order, and the result's own rounding."""
    want, terms = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    return bool(((got.double() - want).abs() <= x.shape[1] * 2.0 ** -24 * terms + rounded * want.abs()).all())


@pytest.mark.parametrize("m,n,k", [
    (17, 24, 512), (33, 1000, 576), (64, 2040, 1024), (65, 136, 512),       # 64 x 64, also of weights with few rows
    (129, 4112, 512), (511, 2072, 2048), (700, 2048, 1088),                 # 128 x 64
    (257, 8200, 2048), (1025, 3080, 1024), (2500, 1032, 576),               # 128 x 128
    (1153, 4104, 576), (2100, 3088, 2048), (2305, 2056, 1024),              # 256 x 128, nine and ten row tiles
    (2047, 4112, 512), (1409, 6152, 1024), (1793, 6144, 640),               # 256 x 192
    (2047, 8192, 576), (1281, 8232, 512),                                   # 256 x 256
    (2048, 8200, 1024), (2635, 6144, 1024)])                                # whole rounds and the rest
def test_products_at_the_edges_of_their_tiles(m, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda").to(bf) for r in (m, n))
    around = torch.full((m + 2, n), 7.0, device="cuda")
    kn.linear(x, w, around[1:-1])
    assert within(around[1:-1], x, w) and bool((around[0] == 7).all()) and bool((around[-1] == 7).all())
    out = torch.full((m, n), float("nan"), dtype=bf, device="cuda")
    kn.linear(x, w, out)
    assert within(out, x, w, 2.0 ** -8)
    pieces = kn.linear_pieces(bf, m, n, k)
    if pieces > 1:
        parts = torch.full((pieces, m, n), float("nan"), device="cuda")
        kn.linear(x, w, parts)
        assert within(parts.double().sum(0), x, w)
    if n % 16 == 0:
        whole, got = torch.empty(m, n, device="cuda"), torch.full((m, n // 2), float("nan"), dtype=bf, device="cuda")
        kn.linear(x, w, whole)
        kn.linear_swiglu(x, w, got, activation="relu")
        gate, up = whole.view(m, n // 16, 2, 8).unbind(2)
        assert torch.equal(got, (gate.clamp(min=0) * up).reshape(m, n // 2).to(bf))


@pytest.mark.parametrize("counts,n,k", [
    ([500, 0, 513, 700, 256, 1, 900, 130], 3584, 576), ([300] * 8, 2048, 512), ([1500, 0, 1200, 5], 5120, 512),
    ([100] * 9, 2056, 1024), ([499] * 8, 3584, 1536)])
def test_groups_of_rows_on_every_tile(counts, n, k):
    """More row tiles than eight over all groups, tiles that end within a group's last rows, empty groups."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    rows = sum(counts) + 19
    x = torch.randn(rows, k, generator=gen, device="cuda").bfloat16()
    x[sum(counts):] = float("nan")
    w = torch.randn(len(counts) * n, k, generator=gen, device="cuda").bfloat16()
    ws = [w[e * n : (e + 1) * n] for e in range(len(counts))]
    out = torch.full((rows, n), 7.0, device="cuda")
    kn.linear_grouped(x, ws, out, torch.tensor(counts, dtype=torch.int32, device="cuda"))
    at = 0
    for e, c in enumerate(counts):
        assert within(out[at : at + c], x[at : at + c], ws[e]), e
        at += c
    assert bool((out[at:] == 7).all())


@pytest.mark.parametrize("n,k", [(128, 512), (1536, 2048), (1000, 4096)])
def test_whole_products_of_a_few_rows_more_than_16(n, k):
    """Up to 32 rows of a narrow weight stay with the kernel of 16 rows: the same sums, bit for bit."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x, w = torch.randn(32, k, generator=gen, device="cuda").bfloat16(), torch.randn(n, k, generator=gen, device="cuda").bfloat16()
    few = torch.cat([kn.linear(x[at : at + 16], w, part := torch.empty(16, n, device="cuda")) or part for at in (0, 16)])
    for rows in (17, 24, 32):
        got = torch.empty(rows, n, device="cuda")
        kn.linear(x[:rows], w, got)
        assert within(got, x[:rows], w) and torch.equal(got, few[:rows])


@pytest.mark.parametrize("n,k", [(2048, 512), (2056, 7296), (4096, 2048), (4104, 1088)])
def test_whole_products_of_13_to_32_rows(n, k):
    """Up to 4 096 columns they stay with the kernel of fewer rows: up to 16 the same sums, bit for bit."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x, w = torch.randn(33, k, generator=gen, device="cuda").to(bf), torch.randn(n, k, generator=gen, device="cuda").to(bf)
    few = torch.empty(12, n, device="cuda")
    kn.linear(x[:12], w, few)
    for held in (w, kn.pack_weight(w)):
        for rows in (13, 16, 17, 32, 33):
            got = torch.full((rows + 1, n), 7.0, device="cuda")
            kn.linear(x[:rows], held, got[:rows])
            assert within(got[:rows], x[:rows], w) and bool((got[rows:] == 7).all())
            assert rows > 16 or n > 4096 or torch.equal(got[:12], few)
            out = torch.full((rows, n), float("nan"), dtype=bf, device="cuda")
            kn.linear(x[:rows], held, out)
            assert torch.equal(out, got[:rows].to(bf))
            if n % 16 == 0:
                gated = torch.full((rows, n // 2), float("nan"), dtype=bf, device="cuda")
                kn.linear_swiglu(x[:rows], held, gated, activation="relu")
                gate, up = got[:rows].view(rows, n // 16, 2, 8).unbind(2)
                assert torch.equal(gated, (gate.clamp(min=0) * up).reshape(rows, n // 2).to(bf))


@pytest.mark.parametrize("m,n,k", [
    (65, 136, 128), (100, 2064, 64), (130, 1000, 320), (300, 28672, 128), (513, 4112, 192), (2049, 6160, 384), (2635, 3072, 320),
    (1025, 8208, 448), (257, 264, 64)])
def test_products_of_a_short_k(m, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda").to(bf) for r in (m, n))
    around = torch.full((m + 2, n), 7.0, device="cuda")
    kn.linear(x, w, around[1:-1])
    assert within(around[1:-1], x, w) and bool((around[0] == 7).all()) and bool((around[-1] == 7).all())
    out = torch.full((m, n), float("nan"), dtype=bf, device="cuda")
    kn.linear(x, w, out)
    assert within(out, x, w, 2.0 ** -8)
    if n % 16 == 0:
        got = torch.full((m, n // 2), float("nan"), dtype=bf, device="cuda")
        kn.linear_swiglu(x, w, got, activation="relu")
        gate, up = (x.double() @ w.double().T).view(m, n // 16, 2, 8).unbind(2)
        off_gate, off_up = (k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).view(m, n // 16, 2, 8).unbind(2)
        want = gate.clamp(min=0) * up
        bound = off_gate * (up.abs() + off_up) + off_up * gate.clamp(min=0) + 2.0 ** -8 * want.abs()
        assert bool(((got.view(m, n // 16, 8).double() - want).abs() <= bound).all())
