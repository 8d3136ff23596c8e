"""All experts' products in one launch against a product an expert, and a mixture of experts whose prompt goes that way against
the way that runs every row through all experts."""
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
            # (each entry: K roundings of 2^-24 of the terms' absolute sum at most, here and in the reference)
            assert ((out[at : at + n] - want).abs() <= 2 * K * 2.0 ** -24 * (x[at : at + n].float().abs() @ w.float().abs().T)).all()
        at += n
    assert (out[total:] == 7.0).all()


@pytest.mark.parametrize("width,inner,more", [
    (512, 576, dict(activation="silu", identity=3, correction=True, shared_inner=512)),
    (576, 512, dict(activation="silu", identity=2, shared_inner=64, shared_gate=True, scoring="softmax", groups=3, keep=2)),
    (512, 512, dict(limit=7.0, weight_input=True)), (512, 520, dict(activation="relu2", identity=1)),
    (640, 512, dict(activation="relu2", correction=True, shared_inner=520))])
def test_a_mixture_sorted_by_expert_in_one_launch(width, inner, more):
    """Sorted and not, the workspace full of NaN: identity experts leave places that no couple takes, and with a correction
    one expert is chosen by nobody."""
    from longbow_quarrel_amd.kernels.hip import HipKernels
    from longbow_quarrel_amd.parts import BuildEnv, StepContext, Workspace
    from longbow_quarrel_amd.parts.feedforward import MixtureOfExperts
    from longbow_quarrel_amd.weights import random_tensors

    kn, dev, rows, E = HipKernels(), torch.device("cuda:0"), 300, 7
    part = MixtureOfExperts(width, E, 3, inner, "m", **{"weight_input": False, "renormalize": True, **more})
    tensors = random_tensors(part.tensor_specs(), 3, torch.bfloat16, 0.05, device=dev)
    tensors["m.router"] = torch.randn_like(tensors["m.router"])
    if part.correction:
        tensors["m.correction"] = torch.zeros(part.outputs, device=dev)
        tensors["m.correction"][2] = -100.0
    part.bind(tensors, BuildEnv(torch.bfloat16, dev, kn))
    h = torch.randn(rows, width, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device=dev)
    got = {}
    for sort in (True, False):
        ws = Workspace(dev, 1 << 27)
        for arena in (ws.step, *ws.runs):
            arena.buf.fill_(255)
        part.sort_from_rows = 256 if sort else rows + 1
        ctx = StepContext(kernels=kn, dtype=torch.bfloat16, device=dev, ws=ws, rows=rows, batch=1, tokens=i32([0] * rows),
                          row_seq=i32([0] * rows), row_pos=i32(range(rows)), seq_slot=i32([0]), seq_start=i32([0]), seq_len=i32([rows]),
                          cu_rows=i32([0, rows]), host_slots=[0], host_start=[0], host_new=[rows], max_new=rows, max_len=rows)
        assert part._sorts(rows, ctx) == sort and (not sort or part._grouped(h, ctx) == (inner % 64 == 0))
        got[sort] = part.forward(h, ctx, out=torch.full((rows, width), float("nan"), device=dev)).float()
        assert ws.fits()
    # Both round an expert's activations to 8 bits from 32-bit sums that may differ in their last: an entry in some 1e4 by
    # 2^-8.  The sums of the last products are of the same terms in another order, within (E inner + 3) 2^-24 of their size.
    assert torch.isfinite(got[True]).all()
    assert (got[True] - got[False]).norm() <= 2e-4 * got[False].norm()
