"""Queries, keys and values of many rows, normed, rotated and stored by runs of rows: the same bits as a few rows at a time."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H,G,more", [
    (64, 5, 2, dict(norm_qk="head", weights=True, dims=64)), (128, 16, 4, dict(norm_qk="head", dims=64, inter=True)),
    (128, 3, 3, dict(bias=True, norm_v=True)), (256, 4, 1, dict(bias=True, norm_qk="head", dims=256, v_from_k=True)),
    (128, 9, 9, dict(norm_qk="head", weights=True, norm_v=True, dims=6)), (64, 1, 17, dict(dims=30, inter=True))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_runs_of_rows(D, H, G, more, dtype):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(D + H)
    dev = lambda *s: torch.randn(*s, generator=gen).cuda()
    lengths, starts = [1, 170, 8, 290, 5, 264], [3, 61, 0, 7, 130, 56]
    rows, BS, slots = sum(lengths), 64, len(lengths)
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lengths)]).int().cuda()
    seq = torch.repeat_interleave(torch.arange(slots), torch.tensor(lengths)).int().cuda()
    slot = torch.randperm(slots, generator=gen).int().cuda()
    table = torch.randperm(slots * 6, generator=gen).int().view(slots, 6).cuda()
    cols = (H + G) * D + (0 if more.get("v_from_k") else G * D)
    src = dev(rows, cols + 4)[:, :cols]
    args = dict(norm_qk=more.get("norm_qk"), norm_v=more.get("norm_v", False), v_from_k=more.get("v_from_k", False))
    if more.get("bias"):
        args["bias"] = dev(cols)
    if more.get("weights"):
        args.update(q_weight=dev(D), k_weight=dev(D))
    angles = None
    if "dims" in more:
        angles = dev(rows, more["dims"] // 2, 2)
        args.update(interleaved=more.get("inter", False), magnitude=1.5)

    def run(lo, hi, q, k, v):
        place = dict(row_pos=pos[lo:hi].contiguous(), row_seq=seq[lo:hi].contiguous(), seq_slot=slot, block_table=table, kcache=k, vcache=v,
                     block_size=BS) if k is not None else {}
        turn = {} if angles is None else {"cos_sin": angles[lo:hi].contiguous()}
        kn.qkv_norm_store(src[lo:hi], q[lo:hi], H, G, D, D, 1e-5, **args, **turn, **place)

    new = lambda: [torch.full((rows, H * D), 7.0, dtype=dtype, device="cuda"), torch.full((slots * 6, G, BS, D), 7.0, dtype=dtype, device="cuda"),
                   torch.full((slots * 6, G, D, BS), 7.0, dtype=dtype, device="cuda")]
    whole, parts, alone = new(), new(), new()
    run(0, rows, *whole)
    for lo in range(0, rows, 50):
        run(lo, min(rows, lo + 50), *parts)
    assert all(torch.equal(a, b) for a, b in zip(whole, parts))
    run(0, rows, alone[0], None, None)
    assert torch.equal(alone[0], whole[0])


@pytest.mark.parametrize("rows,width", [(1, 4), (9, 1024), (3, 1028), (2, 2048), (5, 4096), (130, 3072), (2, 4100)])
@pytest.mark.parametrize("bias", [True, False])
def test_mean_of_normed_branches(rows, width, bias):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator().manual_seed(width)
    stack, w, b = torch.randn(2, rows, width, generator=gen), torch.randn(2, width, generator=gen), torch.randn(2, width, generator=gen)
    out = torch.empty(rows, width, device="cuda")
    kn.rmsnorm_mean(stack.cuda(), [x.cuda() for x in w], 1e-5, out, **({"biases": [b[0].cuda(), None]} if bias else {}))
    y = stack.double()
    if bias:
        y[0] += b[0].double()
    want = (y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-5) * w.double()[:, None]).mean(0)
    size = (y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-5) * w.double()[:, None]).abs().mean(0)
    # (an entry: some ten roundings; the sum of squares: 2^-24 for each of a thread's entries at most, halved by the root)
    assert ((out.cpu().double() - want).abs() <= (16 + width / 256) * 2.0 ** -24 * size + 1e-30).all()


@pytest.mark.parametrize("N,V,H,G,dims,inter", [(64, 64, 3, 2, 64, False), (64, 128, 2, 3, 30, True), (128, 256, 8, 2, 64, False),
                                                (128, 128, 5, 5, 0, False), (256, 512, 2, 1, 256, True), (30, 44, 3, 1, 14, False)])
@pytest.mark.parametrize("rows", [1, 639, 645])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_heads_in_two_parts(N, V, H, G, dims, inter, rows, dtype):
    """Keys of two parts are one row of the cache; otherwise the bits are those of twice as many heads, half as wide."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, M, BS, blocks = HipKernels(), 2, 64, 12
    gen = torch.Generator().manual_seed(N + V + rows)
    pos = torch.arange(5, 5 + rows).int().cuda()
    seq, slot = torch.zeros(rows, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    table = torch.randperm(blocks, generator=gen).int().view(1, blocks).cuda()
    cols = M * (H + G) * N + G * V
    src = torch.randn(rows, (cols + 3) // 4 * 4, generator=gen).cuda()[:, :cols]
    angles = torch.randn(rows, dims // 2, 2, generator=gen).cuda() if dims else None
    made = lambda *s: torch.full(s, 7.0, dtype=dtype, device="cuda")
    q, k, v = made(rows, M * H * N), made(blocks, G, BS, M * N), made(blocks, G, V, BS)
    q2, k2, v2 = made(rows, M * H * N), made(blocks, M * G, BS, N), made(blocks, M * G, V // M, BS)

    def place(lo, hi):
        turn = {} if angles is None else dict(cos_sin=angles[lo:hi].contiguous(), interleaved=inter, magnitude=1.25)
        return dict(row_pos=pos[lo:hi].contiguous(), row_seq=seq[lo:hi].contiguous(), seq_slot=slot, block_table=table, block_size=BS, **turn)

    kn.qkv_norm_store(src, q, H, G, M * N, V, 0.0, maps=M, kcache=k, vcache=v, **place(0, rows))
    for lo in range(0, rows, 100):
        hi = min(rows, lo + 100)
        kn.qkv_norm_store(src[lo:hi], q2[lo:hi], M * H, M * G, N, V // M, 0.0, kcache=k2, vcache=v2, **place(lo, hi))
    assert torch.equal(q, q2) and torch.equal(v, v2.reshape(v.shape))
    assert torch.equal(k, k2.view(blocks, G, M, BS, N).transpose(2, 3).reshape(k.shape))
