"""A feed-forward of two matrices in bfloat16: up to 16 rows its activation lies in the first product's epilogue, beyond it is a kernel of its own."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from longbow_quarrel_amd.parts.feedforward import PlainFeedForward

FORMULAS = {"gelu": F.gelu, "gelu_tanh": lambda v: F.gelu(v, approximate="tanh"), "silu": F.silu, "relu": F.relu, "relu2": lambda v: F.relu(v) ** 2}


@pytest.mark.gpu
@pytest.mark.parametrize("activation", sorted(FORMULAS))
@pytest.mark.parametrize("width,inner", [(512, 2048), (576, 2056), (1024, 4104), (512, 640)])  # (the last: no epilogue for any rows)
@pytest.mark.parametrize("rows", [1, 5, 16, 17])
def test_against_the_formula(activation, width, inner, rows):
    from longbow_quarrel_amd.kernels.hip import HipKernels
    from longbow_quarrel_amd.parts import BuildEnv

    kn, dev = HipKernels(), torch.device("cuda:0")
    assert kn.linear_unit_supported(torch.bfloat16, rows, inner, width, False) == (rows <= 16 and inner >= 2048)
    gen = torch.Generator().manual_seed(width + inner)
    part = PlainFeedForward(width, inner, "m", activation)
    t = {f"m.{n}": (torch.randn(*size, generator=gen) * 0.1).bfloat16().cuda() for n, size in (("up", (inner, width)), ("down", (width, inner)))}
    part.bind(dict(t), BuildEnv(torch.bfloat16, dev, kn))
    h = torch.randn(rows, width, generator=gen).bfloat16().cuda()
    ws = SimpleNamespace(alloc=lambda shape, dtype, **_: torch.full(tuple(shape), float("nan"), dtype=dtype, device=dev))
    got = part.forward(h, SimpleNamespace(kernels=kn, ws=ws, dtype=torch.bfloat16)).double()

    act = FORMULAS[activation](h.double() @ t["m.up"].double().T).bfloat16().double()
    down = t["m.down"].double()
    # 32-bit sums of exact products in the second, and in the first so close to 64 bits that an activation rounds to its other
    # neighbour in bfloat16 (2^-8 of it) about once in a thousand: eight of the row's largest allow for that
    largest = act.abs().amax(1, keepdim=True) * down.abs().amax(1)
    assert ((got - act @ down.T).abs() <= inner * 2.0 ** -24 * (act.abs() @ down.abs().T) + 8 * 2.0 ** -8 * largest).all()
