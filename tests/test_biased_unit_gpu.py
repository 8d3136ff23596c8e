"""A gated unit with biases, whose second product carries its bias as one more column behind the activations."""
from types import SimpleNamespace

import pytest
import torch

from longbow_quarrel_amd.parts.feedforward import GatedLinearUnit


def test_columns_behind_the_activations():
    """K in 128s, which the kernel of at most 8 rows wants, wherever K was in 64s."""
    for inner in (64, 128, 576, 1024, 4032, 7168):
        tail = GatedLinearUnit(64, inner, "m", bias=True).tail
        assert (inner + tail) % 128 == 0 and 0 < tail <= 128
    assert GatedLinearUnit(64, 40, "m", bias=True).tail == 8


@pytest.mark.gpu
@pytest.mark.parametrize("width,inner", [(512, 576), (512, 512), (2048, 640), (264, 520), (2056, 1024)])
@pytest.mark.parametrize("rows", [1, 8, 17, 33, 100])
def test_against_the_formula(width, inner, rows):
    from longbow_quarrel_amd.kernels.hip import HipKernels
    from longbow_quarrel_amd.parts import BuildEnv
    from longbow_quarrel_amd.weights import random_tensors

    kn, dev = HipKernels(), torch.device("cuda:0")
    part = GatedLinearUnit(width, inner, "m", bias=True)
    tensors = random_tensors(part.tensor_specs(), 3, torch.bfloat16, 0.1, device=dev)
    tensors = {s.name: tensors[s.name].float() if s.kind == "vector32" else tensors[s.name] for s in part.tensor_specs()}
    part.bind(dict(tensors), BuildEnv(torch.bfloat16, dev, kn))
    h = torch.randn(rows, width, generator=torch.Generator().manual_seed(inner)).bfloat16().cuda()
    ws = SimpleNamespace(alloc=lambda shape, dtype, **_: torch.full(tuple(shape), float("nan"), dtype=dtype, device=dev))
    got = part.forward(h, SimpleNamespace(kernels=kn, ws=ws, dtype=torch.bfloat16)).double()

    t = {k: v.double() for k, v in tensors.items()}
    g, u = (h.double() @ t[f"m.{n}"].T + t[f"m.{n}.b"] for n in ("gate", "up"))
    act = (g * torch.sigmoid(g) * u).bfloat16().double()
    want = act @ t["m.down"].T + t["m.down.b"]
    # 32-bit sums of exact products in the second, and in the first so close to 64 bits that an activation rounds to its other
    # neighbour in bfloat16 (2^-8 of it) about once in a thousand: four of the row's largest allow for that
    terms = act.abs() @ t["m.down"].abs().T + t["m.down.b"].abs()
    largest = act.abs().amax(1, keepdim=True) * t["m.down"].abs().amax(1)
    assert ((got - want).abs() <= (inner + 128) * 2.0 ** -24 * terms + 4 * 2.0 ** -8 * largest).all()


def bound_part(kn, width, inner, down=torch.bfloat16):
    from longbow_quarrel_amd.parts import BuildEnv
    from longbow_quarrel_amd.weights import random_tensors

    dev = torch.device("cuda:0")
    part = GatedLinearUnit(width, inner, "m", bias=True)
    tensors = random_tensors(part.tensor_specs(), 3, torch.bfloat16, 0.1, device=dev)
    tensors = {s.name: tensors[s.name].float() if s.kind == "vector32" else tensors[s.name] for s in part.tensor_specs()}
    tensors["m.down"] = tensors["m.down"].to(down)
    part.bind(dict(tensors), BuildEnv(torch.bfloat16, dev, kn))
    ws = SimpleNamespace(alloc=lambda shape, dtype, **_: torch.full(tuple(shape), float("nan"), dtype=dtype, device=dev))
    return part, {k: v.double() for k, v in tensors.items()}, SimpleNamespace(kernels=kn, ws=ws, dtype=torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("width,inner", [(512, 1024), (576, 1032), (2048, 1280)])
@pytest.mark.parametrize("rows", [1, 8, 16, 17, 100])
def test_where_the_products_epilogue_applies_the_unit(width, inner, rows):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    part, t, ctx = bound_part(HipKernels(), width, inner)
    assert part.unit
    h = torch.randn(rows, width, generator=torch.Generator().manual_seed(inner)).bfloat16().cuda()
    got = part.forward(h, ctx).double()
    g, u = (h.double() @ t[f"m.{n}"].T + t[f"m.{n}.b"] for n in ("gate", "up"))
    act = (g * torch.sigmoid(g) * u).bfloat16().double()
    want = act @ t["m.down"].T + t["m.down.b"]
    # (the bound of the test above: sums in 32 bits, and four activations that round to their other neighbour)
    terms = act.abs() @ t["m.down"].abs().T + t["m.down.b"].abs()
    largest = act.abs().amax(1, keepdim=True) * t["m.down"].abs().amax(1)
    assert ((got - want).abs() <= (inner + 128) * 2.0 ** -24 * terms + 4 * 2.0 ** -8 * largest).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8, 17, 100])
def test_a_second_matrix_in_32_bits(rows):
    """Its activations stay in 32 bits, so no epilogue rounds them."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    width, inner = 512, 1024
    part, t, ctx = bound_part(HipKernels(), width, inner, torch.float32)
    h = torch.randn(rows, width, generator=torch.Generator().manual_seed(inner)).bfloat16().cuda()
    got = part.forward(h, ctx).double()
    (g, off_g), (u, off_u) = ((h.double() @ t[f"m.{n}"].T + t[f"m.{n}.b"],
                               (h.double().abs() @ t[f"m.{n}"].abs().T + t[f"m.{n}.b"].abs()) * (width + 1) * 2.0 ** -24) for n in ("gate", "up"))
    silu = g * torch.sigmoid(g)
    # an activation is off by what its sums are (silu' is below 1.1) and a few roundings; then come `inner` terms
    off = 1.1 * off_g * (u.abs() + off_u) + silu.abs() * off_u + 8 * 2.0 ** -24 * (silu * u).abs()
    down, bias = t["m.down"].T, t["m.down.b"]
    terms = (silu * u).abs() @ down.abs() + bias.abs()
    assert ((got - (silu * u) @ down - bias).abs() <= 1.01 * (off @ down.abs() + (inner + 128) * 2.0 ** -24 * terms)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 5, 16, 40])
@pytest.mark.parametrize("row,first", [(513, 1), (512, 4), (516, 0)])
def test_rows_at_any_address_with_dense_weights(rows, row, first):
    """Rows that begin at no multiple of 16 bytes: as the same rows side by side, but for the order of sums."""
    from longbow_quarrel_amd.kernels.hip import HipKernels
    from longbow_quarrel_amd.parts import BuildEnv
    from longbow_quarrel_amd.parts.feedforward import PlainFeedForward

    kn, width, inner = HipKernels(), 512, 2048
    kn.pack_weights = False
    gen = torch.Generator().manual_seed(rows + row)
    apart = torch.randn(rows * row + 8, generator=gen).bfloat16().cuda()[first:].as_strided((rows, width), (row, 1))
    gated, _, ctx = bound_part(kn, width, inner)
    plain = PlainFeedForward(width, inner, "m", "relu2")
    plain.bind({f"m.{n}": (torch.randn(*size, generator=gen) * 0.1).bfloat16().cuda() for n, size in
                (("up", (inner, width)), ("down", (width, inner)))}, BuildEnv(torch.bfloat16, torch.device("cuda:0"), kn))
    assert gated.unit
    for part in (gated, plain):
        want, got = part.forward(apart.clone(memory_format=torch.contiguous_format), ctx).double(), part.forward(apart, ctx).double()
        # an activation whose sum lies next to the middle between two bfloat16 numbers may round to the other one, 2^-8 of it: one in
        # hundreds, so that a result of some thousand terms with signs is off by far less than its row's norm times 2^-8
        assert ((got - want).norm(dim=1) <= 2.0 ** -8 * want.norm(dim=1)).all()
