"""What stands between a layer's first products and its attention, against the formulas in 64 bits: queries, keys and values (few
rows and many, whole heads and heads in parts), and a latent layer's rows and queries."""
import pytest
import torch

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def turned(x, angles, dims, interleaved, magnitude):
    """The first `dims` entries of x [..., n] rotated by angles [..., pairs, 2] -> (result, size of its terms)."""
    c, s = angles[..., 0] * magnitude, angles[..., 1] * magnitude
    head, rest = x[..., :dims], x[..., dims:]
    a, b = (head[..., 0::2], head[..., 1::2]) if interleaved else head.chunk(2, -1)
    new, size = (a * c - b * s, b * c + a * s), ((a * c).abs() + (b * s).abs(), (b * c).abs() + (a * s).abs())
    join = lambda p: torch.stack(p, -1).flatten(-2) if interleaved else torch.cat(p, -1)
    return torch.cat([join(new), rest], -1), torch.cat([join(size), rest.abs()], -1)


def normed(x, size, eps, w=None):
    factor = 1 / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 if w is None else w)
    return x * factor, size * factor.abs()


def close(got, want, size):
    """Some thirty roundings on the way (cos, sin, products, the norm's root and the half of its sum's, the weight), and the result's."""
    out = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2 * U
    return bool(((got.double() - want).abs() <= 32 * U * size + out * want.abs()).all())


def placed(lengths, starts, BS, gen):
    """Rows of sequences at their positions: row_pos, row_seq, slots, table, and for every row its block and offset."""
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lengths)])
    seq = torch.repeat_interleave(torch.arange(len(lengths)), torch.tensor(lengths))
    slot, per = torch.randperm(len(lengths), generator=gen), max(s + n for s, n in zip(starts, lengths)) // BS + 1
    table = torch.randperm(len(lengths) * per, generator=gen).view(len(lengths), per)
    block = table[slot[seq], pos // BS]
    i32 = lambda t: t.int().cuda()
    return dict(row_pos=i32(pos), row_seq=i32(seq), seq_slot=i32(slot), block_table=i32(table)), block.cuda(), (pos % BS).cuda(), table.numel()


@pytest.mark.parametrize("D,V,H,G,maps,more", [
    (64, 64, 5, 2, 1, dict(norm="head", weights=True, dims=64, inter=True, bias=True)), (128, 128, 3, 3, 1, dict(norm_v=True, dims=64, bias=True)),
    (256, 256, 4, 2, 1, dict(norm="head", dims=30, from_k=True, bias=True)), (256, 256, 3, 2, 2, dict(dims=64)),
    (128, 128, 4, 2, 2, dict(dims=64, inter=True, norm="head", weights=True)), (48, 40, 3, 1, 1, dict(norm="row", weights=True))])
@pytest.mark.parametrize("lengths,starts", [([1, 4, 2], [63, 0, 130]), ([1, 250, 9, 1900], [7, 60, 0, 131])])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_queries_keys_and_values(D, V, H, G, maps, more, lengths, starts, dtype):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, BS, rows, eps, mag = HipKernels(), 64, sum(lengths), 1e-5, 1.25
    gen = torch.Generator().manual_seed(D + H + rows)
    dev = lambda *s: torch.randn(*s, generator=gen).cuda()
    place, block, off, blocks = placed(lengths, starts, BS, gen)
    from_k, dims, norm, unit = more.get("from_k", False), more.get("dims", 0), more.get("norm"), D // maps
    cols = (H + G) * D + (0 if from_k else G * V)
    src = dev(rows, (cols + 7) // 4 * 4)[:, :cols]
    args = dict(norm_qk=norm, norm_v=more.get("norm_v", False), v_from_k=from_k, maps=maps, **place)
    if more.get("bias"):
        args["bias"] = dev(cols)
    if more.get("weights"):
        args.update(q_weight=dev(H * D if norm == "row" else unit), k_weight=dev(G * D if norm == "row" else unit))
    if dims:
        args.update(cos_sin=dev(rows, dims // 2, 2), interleaved=more.get("inter", False), magnitude=mag)
    made = lambda *s: torch.full(s, 7.0, dtype=dtype, device="cuda")
    q, k, v = made(rows, H * D), made(blocks, G, BS, D), made(blocks, G, V, BS)
    kn.qkv_norm_store(src, q, H, G, D, V, eps, kcache=k, vcache=v, block_size=BS, **args)

    x = src.double() + (args["bias"].double() if "bias" in args else 0.0)
    row_wise = norm == "row"

    def unit_of(part, heads, w):
        y = part.reshape(rows, 1, heads * D) if row_wise else part.reshape(rows, heads * maps, unit)
        size = y.abs()
        if dims:
            y, size = turned(y, args["cos_sin"].double()[:, None], dims, args["interleaved"], mag)
        if norm:
            y, size = normed(y, size, eps, w if w is None else w.double())
        return y.reshape(rows, heads, D), size.reshape(rows, heads, D)

    want, size = unit_of(x[:, : H * D], H, args.get("q_weight"))
    assert close(q.view(rows, H, D), want, size)
    keys = x[:, H * D : (H + G) * D]
    want, size = unit_of(keys, G, args.get("k_weight"))
    assert close(k[block, :, off], want, size)
    want = (keys if from_k else x[:, (H + G) * D :]).reshape(rows, G, V)
    size = want.abs()
    if args["norm_v"]:
        want, size = normed(want, size, eps)
    assert close(v[block, :, :, off], want, size)
    k[block, :, off], v[block, :, :, off] = 7.0, 7.0
    assert bool((k == 7).all()) and bool((v == 7).all())  # (nothing beside the rows' places)


@pytest.mark.parametrize("heads,dim,rd,dims,rank,qr,inter", [
    (1, 16, 2, 2, 1, 1, False), (16, 128, 64, 64, 192, 768, True), (3, 48, 10, 6, 65, 257, False), (2, 64, 8, 8, 2048, 100, False)])
@pytest.mark.parametrize("lengths,starts", [([1], [64]), ([9, 7], [60, 0]), ([30, 100], [130, 1])])
def test_a_latent_layers_rows_and_queries(heads, dim, rd, dims, rank, qr, inter, lengths, starts):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, BS, rows, eps, mag = HipKernels(), 64, sum(lengths), 1e-5, 1.25
    gen = torch.Generator().manual_seed(rows + rank)
    dev = lambda *s: torch.randn(*s, generator=gen).cuda()
    place, block, off, blocks = placed(lengths, starts, BS, gen)
    kd = rank + rd
    src, wq, wkv, angles = dev(rows, 8 + qr + kd)[:, 8:], dev(qr), dev(rank), dev(rows, dims // 2, 2)
    bf = lambda *s: torch.full(s, 7.0, dtype=torch.bfloat16, device="cuda")
    cq, k, v = bf(rows, qr), bf(blocks, 1, BS, kd), bf(blocks, 1, rank, BS)
    turn = dict(rot_dim=rd, cos_sin=angles, interleaved=inter, magnitude=mag)
    kn.latent_rows(src, wq, cq, eps, kv_weight=wkv, kcache=k, vcache=v, block_size=BS, **turn, **place)
    x = src.double()
    assert close(cq, *normed(x[:, :qr], x[:, :qr].abs(), eps, wq.double()))
    latent = normed(x[:, qr : qr + rank], x[:, qr : qr + rank].abs(), eps, wkv.double())
    rotated = turned(x[:, qr + rank :], angles.double(), dims, inter, mag)
    assert close(k[block, 0, off], *(torch.cat(p, -1) for p in zip(latent, rotated))) and close(v[block, 0, :, off], *latent)
    k[block, :, off], v[block, :, :, off] = 7.0, 7.0
    assert bool((k == 7).all()) and bool((v == 7).all())

    wide = heads * (dim + rd)
    x, w = dev(rows, (wide + 7) // 4 * 4)[:, :wide], dev(heads, rank, dim).bfloat16()
    q = bf(rows, heads * kd)
    kn.latent_query(x, w, q, **turn)
    plain = x[:, : heads * dim].bfloat16().double().reshape(rows, heads, dim)
    want = torch.einsum("rhd,hkd->rhk", plain.cpu(), w.double().cpu()).cuda()
    size = torch.einsum("rhd,hkd->rhk", plain.abs().cpu(), w.double().abs().cpu()).cuda() * dim / 32  # (a rounding a term)
    rot, rsize = turned(x[:, heads * dim :].double().reshape(rows, heads, rd), angles.double()[:, None], dims, inter, mag)
    assert close(q.view(rows, heads, kd), torch.cat([want, rot], -1), torch.cat([size + want.abs(), rsize], -1))
