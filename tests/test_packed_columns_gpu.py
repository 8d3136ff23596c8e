"""Runs of a packed weight's columns, as a mixture's experts have them: products against 64 bits, and a mixture whose second
matrix is packed against one whose is dense."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N, K, E = 2056, 576, 4


def within(got, x, w):
    """Products of bfloat16 are exact in 32 bits: at most K roundings of 2^-24 of the terms' absolute sum, in any order."""
    want, terms = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    return bool(((got.double() - want).abs() <= x.shape[1] * 2.0 ** -24 * terms).all())


@pytest.fixture(scope="module")
def held():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    whole = torch.randn(N, E * K, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").bfloat16()
    packed = kn.pack_weight(whole)
    ws = [kn.weight_columns(packed, e * K, K) for e in range(E)]
    assert packed is not whole and all(w.packed and not w.is_contiguous() for w in ws)
    return kn, whole, ws


@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 40, 64, 65, 300, 2100])
def test_products(held, rows):
    kn, whole, ws = held
    x = torch.randn(rows, K, generator=torch.Generator(device="cuda").manual_seed(rows), device="cuda").bfloat16()
    for e in (0, E - 1):
        dense = whole[:, e * K : (e + 1) * K]
        got = torch.full((rows + 1, N), 7.0, device="cuda")
        kn.linear(x, ws[e], got[:rows])
        assert within(got[:rows], x, dense) and bool((got[rows] == 7).all())
        pieces = kn.linear_pieces(torch.bfloat16, rows, N, K)
        parts = torch.full((pieces, rows, N), float("nan"), device="cuda")
        kn.linear(x, ws[e], parts)
        assert within(parts.double().sum(0), x, dense)


@pytest.mark.parametrize("counts", [  # 128 x 128, 256 x 128, 256 x 192 and 256 x 256 tiles
    [300, 0, 129, 271], [700, 513, 0, 790], [1500, 1, 1023, 1480], [3000, 0, 1, 3001]])
def test_products_of_all_experts(held, counts):
    kn, whole, ws = held
    total = sum(counts)
    x = torch.randn(total + 37, K, generator=torch.Generator(device="cuda").manual_seed(total), device="cuda").bfloat16()
    x[total:] = float("nan")
    out = torch.full((total + 37, N), 7.0, device="cuda")
    kn.linear_grouped(x, ws, out, torch.tensor(counts, dtype=torch.int32, device="cuda"))
    at = 0
    for e, n in enumerate(counts):
        if n:
            assert within(out[at : at + n], x[at : at + n], whole[:, e * K : (e + 1) * K])
        at += n
    assert bool((out[total:] == 7).all())


@pytest.mark.parametrize("more", [dict(activation="silu", shared_inner=512), dict(limit=7.0, weight_input=True),
                                  dict(activation="relu2", identity=1)])
def test_a_mixture(more):
    """The same bits with its matrices packed and dense: every way that a step's rows can take (the chosen experts alone, all
    experts' columns, sorted by expert)."""
    from longbow_quarrel_amd.kernels.hip import HipKernels
    from longbow_quarrel_amd.parts import BuildEnv, StepContext, Workspace
    from longbow_quarrel_amd.parts.feedforward import MixtureOfExperts
    from longbow_quarrel_amd.weights import random_tensors

    dev, width = torch.device("cuda:0"), 2048
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device=dev)
    results = {}
    for pack in (True, False):
        kn = HipKernels()
        kn.pack_weights = pack
        part = MixtureOfExperts(width, 5, 2, 512, "m", **{"weight_input": False, "renormalize": True, **more})
        tensors = random_tensors(part.tensor_specs(), 3, torch.bfloat16, 0.05, device=dev)
        tensors["m.router"] = torch.randn(tensors["m.router"].shape, generator=torch.Generator().manual_seed(5)).bfloat16().to(dev)
        part.bind(tensors, BuildEnv(torch.bfloat16, dev, kn))
        assert bool(getattr(part.w_down, "packed", False)) == pack and part.down_of[1].is_contiguous() is False
        for rows in (1, 8, 16, 17, 100, 300):
            h = torch.randn(rows, width, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
            ws = Workspace(dev, 1 << 27)
            for arena in (ws.step, *ws.runs):
                arena.buf.fill_(255)
            ctx = StepContext(kernels=kn, dtype=torch.bfloat16, device=dev, ws=ws, rows=rows, batch=1, tokens=i32([0] * rows),
                              row_seq=i32([0] * rows), row_pos=i32(range(rows)), seq_slot=i32([0]), seq_start=i32([0]),
                              seq_len=i32([rows]), cu_rows=i32([0, rows]), host_slots=[0], host_start=[0], host_new=[rows],
                              max_new=rows, max_len=rows)
            got = part.forward(h, ctx, out=torch.full((rows, width), float("nan"), device=dev)).clone()
            assert torch.isfinite(got).all() and part._few(h, ctx) == (rows <= 16) and part._sorts(rows, ctx) == (rows >= 256)
            results[pack, rows] = got
    for rows in (1, 8, 16, 17, 100, 300):
        assert torch.equal(results[True, rows], results[False, rows]), rows
