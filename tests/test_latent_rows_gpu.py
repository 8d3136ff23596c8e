"""A latent layer's norms, rotations, store and fold in two launches, against the launches that make them one by one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,heads,dim,rd,dims,rank,qr,inter", [
    (1, 1, 16, 2, 2, 1, 1, False), (8, 16, 128, 64, 64, 192, 768, True), (65, 3, 48, 10, 6, 65, 257, False),
    (130, 5, 32, 64, 30, 128, 2048, True), (64, 2, 64, 8, 8, 2048, 100, False), (3, 32, 128, 64, 64, 192, 1536, True)])
@pytest.mark.parametrize("own", [True, False])
def test_rows_and_queries(rows, heads, dim, rd, dims, rank, qr, inter, own):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    assert kn.latent_accepts(torch.bfloat16, heads, dim, rd, rank, qr)
    gen = torch.Generator().manual_seed(rows + rank)
    dev = lambda *s: torch.randn(*s, generator=gen).cuda()
    kd, batch, BS, mag = rank + rd, 2, 64, 1.25
    src = dev(rows, 8 + qr + kd)[:, 8 : 8 + qr + (kd if own else 0)]  # (a run of columns of a wider row)
    wq, wkv, eps = dev(qr), dev(rank), 1e-5
    first = (rows + 1) // 2
    pos = torch.cat([torch.arange(first) + 60, torch.arange(rows - first)]).int().cuda()
    seq = (torch.arange(rows) >= first).int().cuda()
    slot = torch.tensor([2, 0], dtype=torch.int32).cuda()
    blocks = (max(rows, 64) + 60) // BS + 1
    table = torch.randperm(3 * blocks, generator=gen).int().view(3, blocks).cuda()
    freqs = (10000.0 ** (-torch.arange(dims // 2, dtype=torch.float64) / max(1, dims // 2))).cuda()
    angles = torch.empty(rows, dims // 2, 2, device="cuda")
    kn.rope_table(freqs, pos, angles)

    bf = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    cq, want_cq = bf(rows, qr), bf(rows, qr)
    k, v, want_k, want_v = bf(3 * blocks, 1, BS, kd), bf(3 * blocks, 1, rank, BS), bf(3 * blocks, 1, BS, kd), bf(3 * blocks, 1, rank, BS)
    turn = dict(rot_dim=rd, cos_sin=angles, interleaved=inter, magnitude=mag)
    kn.rmsnorm_cols(src[:, :qr], wq, eps, want_cq)
    more = {}
    if own:
        row = bf(rows, kd)
        kn.rmsnorm_cols(src[:, qr : qr + rank], wkv, eps, row[:, :rank])
        kn.rotary(src[:, qr + rank :], row[:, rank:], 1, rd, rd, dims, inter, freqs, mag, pos)
        kn.kv_store(row, row[:, :rank], 1, kd, rank, pos, seq, slot, table, want_k, want_v, BS)
        more = dict(turn, kv_weight=wkv, row_pos=pos, row_seq=seq, seq_slot=slot, block_table=table, kcache=k, vcache=v, block_size=BS)
    kn.latent_rows(src, wq, cq, eps, **more)

    x, w = dev(rows, heads * (dim + rd) + 4)[:, : heads * (dim + rd)] if heads * (dim + rd) % 4 == 0 else dev(rows, heads * (dim + rd) + 4 - heads * (dim + rd) % 4)[:, : heads * (dim + rd)], dev(heads, rank, dim).bfloat16()
    q, want_q = bf(rows, heads * kd), bf(rows, heads * kd)
    kn.latent_query(x, w, q, **turn)
    kn.linear_heads(x[:, : heads * dim].bfloat16().contiguous(), w, want_q, heads, kd)
    kn.rotary(x[:, heads * dim :], want_q[:, rank:], heads, rd, kd, dims, inter, freqs, mag, pos)
    # the same sums in the same order; a contraction more or less may move a result to the next of bfloat16's numbers
    for got, want in ((cq, want_cq), (k, want_k), (v, want_v), (q, want_q)):
        assert ((got.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 1e-6).all()


def test_sizes_that_are_not_taken():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    assert not kn.latent_accepts(torch.float32, 1, 16, 2, 1, 1)
    for sizes in ((1, 24, 2, 1, 1), (1, 16, 2, 2049, 1), (1, 16, 2, 1, 2049), (1, 16, 1025, 1, 1)):
        assert not kn.latent_accepts(torch.bfloat16, *sizes)
