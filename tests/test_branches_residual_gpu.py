"""The norm of one sublayer's result, whole or in pieces, and of the mean of several, added to the stream: against 64 bits, few and
many rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def normed(y, w, eps):
    return y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps) * w


def close(got, x, y, w, roundings):
    """got = x + N(sum of y) w.  The sum's error, 2^-24 of its terms' size for each rounding that they saw, is multiplied by the norm;
    the normed part has some ten roundings and its sum of squares 2^-24 for each of a thread's entries at most (half of that behind
    the root); the result has its own."""
    whole = y.sum(0)
    factor = w.abs() / torch.sqrt((whole * whole).mean(-1, keepdim=True) + 1e-5)
    want = x + normed(whole, w, 1e-5)
    u = 2.0 ** -24
    bound = u * (roundings * y.abs().sum(0) * factor + (16 + got.shape[1] / 256) * whole.abs() * factor + 2 * want.abs())
    return bool(((got.double() - want).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("pieces", [None, 1, 2, 4])
@pytest.mark.parametrize("rows,width", [(1, 4), (3, 1028), (9, 2048), (513, 2052), (2, 3072), (600, 4096), (5, 4100), (520, 8192)])
@pytest.mark.parametrize("rounded", [None, torch.bfloat16, torch.float32])
def test_a_norm_onto_the_stream(rows, width, pieces, rounded):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(rows + width)
    x, w = torch.randn(rows, width, generator=gen), torch.randn(width, generator=gen)
    y = torch.randn(pieces or 1, rows, width, generator=gen)
    got = x.cuda()
    copy = None if rounded is None else torch.empty(rows, width, dtype=rounded, device="cuda")
    kn.rmsnorm_residual(got, (y if pieces else y[0]).contiguous().cuda(), w.cuda(), 1e-5, rounded=copy)
    assert close(got.cpu(), x.double(), y.double(), w.double(), pieces or 1)
    if rounded is not None:
        assert torch.equal(copy, got.to(rounded))


@pytest.mark.parametrize("rows,width,n", [(1, 1024, 2), (8, 4096, 2), (600, 4096, 3), (513, 3072, 2), (530, 2048, 4), (7, 2052, 1), (515, 8192, 2)])
def test_a_mean_of_branches_onto_the_stream(rows, width, n):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(rows + width)
    x, w = torch.randn(rows, width, generator=gen), torch.randn(width, generator=gen)
    stack, ws, bias = torch.randn(n, rows, width, generator=gen), torch.randn(n, width, generator=gen), torch.randn(width, generator=gen)
    got = x.cuda()
    kn.mean_residual(got, stack.cuda(), [v.cuda() for v in ws], [bias.cuda()] + [None] * (n - 1), 1e-5, w.cuda(), 1e-5)
    y = stack.double()
    y[0] += bias.double()
    y = normed(y, ws.double()[:, None], 1e-5) / n
    # (a branch is normed like the sum is: its entries come with 16 + width / 256 roundings)
    assert close(got.cpu(), x.double(), y, w.double(), n + 16 + width / 256)


def test_pieces_of_a_width_that_goes_another_way():
    from longbow_quarrel_amd.kernels.hip import HipKernels, KernelLibraryError

    kn = HipKernels()
    for width in (6, 8196):
        x, w = torch.ones(2, width, device="cuda"), torch.ones(width, device="cuda")
        with pytest.raises(KernelLibraryError):
            kn.rmsnorm_residual(x, torch.ones(2, 2, width, device="cuda"), w, 1e-5)
        assert not kn.mean_residual_takes(width) and bool((x == 1).all())
