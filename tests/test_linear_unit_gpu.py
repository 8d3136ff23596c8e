"""The first product of a feed-forward with its activation in the epilogue: gated silu with biases and the columns behind it at the
edges of every kernel and tile, and plain activations of few rows, against the product and the activation kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(rows, n, k):
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda").bfloat16() for r in (rows, n))
    return x, w * 0.05, torch.randn(n, generator=gen, device="cuda")


@pytest.mark.parametrize("rows,n,k,tail", [
    (1, 2048, 512, 8), (8, 2064, 1024, 128), (16, 28672, 576, 64), (17, 2048, 512, 8), (64, 4112, 640, 128), (65, 2064, 512, 128),
    (130, 4096, 1088, 0), (300, 8208, 512, 8), (1025, 3088, 512, 128), (1409, 6160, 576, 64), (2047, 8208, 512, 128), (2048, 14336, 2048, 128)])
def test_gated_with_biases(rows, n, k, tail):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    x, w, bias = operands(rows, n, k)
    inner = n // 2
    assert kn.linear_unit_supported(bf, rows, n, k, True)
    product = torch.empty(rows, n, device="cuda")
    kn.linear(x, w, product)
    both = torch.cat([part.reshape(rows, inner) for part in (product + bias).view(rows, n // 16, 2, 8).unbind(2)], dim=1).contiguous()
    want = torch.empty(rows, inner + tail, dtype=bf, device="cuda")
    kn.glu(both, want, "silu", tail=tail)
    for held in (w, kn.pack_weight(w)):
        wide = torch.full((rows + 1, inner + tail + 3), 7.0, dtype=bf, device="cuda")
        for out in (torch.empty_like(want), wide[:rows, 1 : inner + tail + 1]):
            kn.linear_unit(x, held, out, "silu", bias=bias, tail=tail)
            # (the exponential and the reciprocal of the hardware: a result may round to the neighbour, 2^-7 of it at most; a product
            # whose gate is far below zero, or whose parts nearly cancel, is off by roundings of 2^-24 of its terms)
            assert ((out.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 1e-5).all()
            assert torch.equal(out[:, inner:], want[:, inner:])
        assert bool((wide[:, 0] == 7).all()) and bool((wide[:, inner + tail + 1 :] == 7).all()) and bool((wide[rows] == 7).all())


@pytest.mark.parametrize("rows,n,k,tail", [
    (4, 2048, 1024, 8), (2, 2048, 8192, 128), (8, 2048, 4096, 8), (8, 2064, 1024, 128), (40, 14336, 2048, 8), (65, 2064, 512, 128), (300, 8208, 512, 8), (2047, 8208, 512, 128), (2048, 14336, 2048, 128)])
def test_gated_with_biases_has_the_activation_kernels_bits(rows, n, k, tail):
    """Sizes whose sums are made in one order either way: the epilogue's functions are then as exact as the activation kernel's."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, inner = HipKernels(), n // 2
    x, w, bias = operands(rows, n, k)
    product = torch.empty(rows, n, device="cuda")
    kn.linear(x, w, product)
    both = torch.cat([part.reshape(rows, inner) for part in (product + bias).view(rows, n // 16, 2, 8).unbind(2)], dim=1).contiguous()
    want = torch.empty(rows, inner + tail, dtype=torch.bfloat16, device="cuda")
    kn.glu(both, want, "silu", tail=tail)
    for held in (w, kn.pack_weight(w)):
        out = torch.empty_like(want)
        kn.linear_unit(x, held, out, "silu", bias=bias, tail=tail)
        assert torch.equal(out, want)


@pytest.mark.parametrize("activation", ["silu", "relu", "gelu_tanh", "gelu", "relu2"])
@pytest.mark.parametrize("rows,n,k", [(1, 2048, 512), (7, 2056, 2048), (16, 10752, 576)])
def test_plain_activations_of_few_rows(activation, rows, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    x, w, _ = operands(rows, n, k)
    assert kn.linear_unit_supported(bf, rows, n, k, False) and not kn.linear_unit_supported(bf, 17, n, k, False)
    for held in (w, kn.pack_weight(w)):
        got, whole = torch.empty(rows, n, dtype=bf, device="cuda"), torch.empty(rows, n, device="cuda")
        kn.linear_unit(x, held, got, activation)
        want = (x.double() @ w.double().T).float()
        exact = torch.empty(rows, n, dtype=bf, device="cuda")
        kn.activation(want, exact, activation)
        # sums in another order: roundings of 2^-24 a term, at most 1.13 (relu2: twice the result) times as large behind the activation,
        # and the result's own rounding
        terms = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        slope = 2 * (want.double().abs() + terms) if activation == "relu2" else 1.13
        assert ((got.double() - exact.double()).abs() <= slope * terms + 2.0 ** -7 * exact.double().abs()).all()


def test_what_is_not_taken():
    from longbow_quarrel_amd.kernels.hip import HipKernels, KernelLibraryError

    kn, bf = HipKernels(), torch.bfloat16
    for size in ((4, 2040, 512, True), (4, 2056, 512, True), (4, 2048, 520, True), (4, 2048, 448, False)):
        assert not kn.linear_unit_supported(bf, *size)
    assert not kn.linear_unit_supported(torch.float32, 4, 2048, 512, True)
    x, w, bias = operands(4, 2048, 512)
    out = torch.empty(4, 1024 + 8, dtype=bf, device="cuda")
    for bad in (dict(activation="relu", bias=bias, tail=8), dict(activation="silu", bias=bias, tail=0), dict(activation="silu", bias=bias[:-1], tail=8)):
        with pytest.raises(KernelLibraryError):
            kn.linear_unit(x, w, out, **bad)
