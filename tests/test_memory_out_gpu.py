"""The matrix memory's answer at heads of every length around a wavefront's runs of 64 entries."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 2, 63, 64, 65, 128, 129, 511, 512, 513, 700])
@pytest.mark.parametrize("rows,heads", [(1, 1), (3, 5)])
def test_memory_out(P, rows, heads):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, scale, eps0, eps = HipKernels(), 0.25, 1e-4, 1e-3
    gen = torch.Generator().manual_seed(P + rows)
    y, z = torch.randn(rows, heads, P + 1, generator=gen), torch.randn(rows, heads, P, generator=gen)
    floor, w = torch.rand(rows, heads, generator=gen), torch.randn(heads, P, generator=gen)
    o = scale * y[..., :P].double() / (torch.maximum((scale * y[..., P].double()).abs(), floor.double()) + eps0)[..., None]
    want = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * w.double() * torch.sigmoid(z.double())
    for dtype, ulp in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)):
        out = torch.full((rows, heads * P + 3), 7.0, dtype=dtype, device="cuda")
        kn.memory_out(y.reshape(rows, -1).cuda(), floor.cuda(), z.reshape(rows, -1).cuda(), w.reshape(-1).cuda(), scale, eps0, eps,
                      out[:, : heads * P])
        # (an entry: some twenty roundings, the exponential's few among them; the sum of squares: one for each of a lane's entries)
        bound = (32 + P / 64) * 2.0 ** -24 * want.abs() * (1 + z.abs()) + ulp * want.abs() + 1e-30
        assert ((out[:, : heads * P].cpu().double().view(rows, heads, P) - want).abs() <= bound).all()
        assert bool((out[:, heads * P :] == 7.0).all())
