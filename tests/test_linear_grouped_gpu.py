"""All experts' products in one launch against a product an expert: the rows' sums are the same, in the same order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,N,K,columns", [
    ([1, 0, 128, 129], 256, 512, False), ([127, 0, 0, 1], 136, 512, True), ([0, 300], 2048, 512, False),
    ([257, 256, 0, 600], 256, 576, True), ([300, 511, 513], 2056, 512, False), ([0, 0], 128, 512, True),
    ([5] * 64, 64, 512, True)])
def test_grouped_products(counts, N, K, columns):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(sum(counts) + N)
    E, total = len(counts), sum(counts)
    rows = total + 37  # (places that no couple takes: what lies there is neither read nor written)
    x = torch.randn(rows, K, generator=gen).bfloat16().cuda()
    x[total:] = float("nan")
    if columns:
        whole = torch.randn(N, E * K, generator=gen).bfloat16().cuda()
        ws = [whole[:, e * K : (e + 1) * K] for e in range(E)]
    else:
        whole = torch.randn(E * N, K, generator=gen).bfloat16().cuda()
        held = kn.pack_weight(whole)
        ws = [kn.weight_rows(held, e * N, N) for e in range(E)]
        assert all(w is not None for w in ws)
    assert kn.linear_grouped_supported(torch.bfloat16, E, N, K)
    assert not kn.linear_grouped_supported(torch.float32, E, N, K) and not kn.linear_grouped_supported(torch.bfloat16, 65, N, K)
    out = torch.full((rows, N), 7.0, device="cuda")
    kn.linear_grouped(x, ws, out, torch.tensor(counts, dtype=torch.int32, device="cuda"))
    at = 0
    for e, n in enumerate(counts):
        if n:
            w = whole[:, e * K : (e + 1) * K] if columns else whole[e * N : (e + 1) * N]
            want = x[at : at + n].float() @ w.float().T  # (products of bfloat16 are exact: 32-bit sums of K terms)
            assert (out[at : at + n] - want).abs().max() <= 2 * K * 2.0 ** -24 * (x[at : at + n].float().abs() @ w.float().abs().T).max()
        at += n
    assert (out[total:] == 7.0).all()
