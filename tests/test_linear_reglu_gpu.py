"""The product that leaves relu(gate) * up, in every kernel that has the epilogue, against 64-bit sums of the same inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m", [1, 8, 17, 33, 64, 65, 300, 2048])
@pytest.mark.parametrize("inner,k", [(8, 8), (328, 96), (1000, 264), (7168, 512), (4096, 512)])
def test_relu_of_gate_times_up(m, inner, k, packed):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    g = torch.Generator().manual_seed(m + inner)
    x, gate, up = (torch.randn(*s, generator=g).bfloat16() for s in ((m, k), (inner, k), (inner, k)))
    w = kn.interleave_gate_up(gate.cuda(), up.cuda())
    if packed:
        w = kn.pack_weight(w)
        if not getattr(w, "packed", False):
            pytest.skip("a weight of this size is not packed")
    out = torch.full((m + 1, inner), 7.0, dtype=torch.bfloat16, device="cuda")  # (a row too many: it stays as it is)
    kn.linear_swiglu(x.cuda(), w, out[:m], activation="relu")
    got = out.cpu().double()
    a, b = x.double() @ gate.double().t(), x.double() @ up.double().t()
    # sums of k terms in 32 bits: each within k 2^-24 of the sum of the terms' sizes; the result is rounded to 8 bits
    da, db = (k * 2.0 ** -24 * (x.double().abs() @ v.double().abs().t()) for v in (gate, up))
    want = a.clamp(min=0) * b
    bound = (da * b.abs() + db * a.abs() + da * db) * 1.01 + 2.0 ** -8 * (want.abs() + da * b.abs() + db * a.abs())
    assert bool(((got[:m] - want).abs() <= bound + 1e-30).all())
    assert bool((got[m] == 7.0).all())
