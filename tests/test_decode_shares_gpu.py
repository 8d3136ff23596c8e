"""Decoding attention at the lengths where cache blocks, takes of several blocks, whole rows and shares of a row end, and with operands
that do not lie on 16 bytes, against the plain implementation in float64."""
import math

import pytest
import torch

from test_kernels_gpu import BS, DEV, i32, kn, paged_cache, rel_err, run_attention  # noqa: F401
import plain

pytestmark = pytest.mark.gpu

EDGES = [1, 63, 64, 65, 128, 129, 192, 193, 256, 257, 384, 385, 386, 640, 1030, 2049]


@pytest.mark.parametrize("heads,kv_heads,head_dim,rows", [(32, 8, 128, 3), (16, 16, 64, 16), (8, 1, 64, 1), (6, 2, 256, 4),
                                                          (4, 1, 192, 16), (64, 32, 64, 16), (48, 48, 128, 14)])
@pytest.mark.parametrize("window", [0, 70])
@pytest.mark.parametrize("apart", [0, 1])
def test_folded_rows_at_the_edges(kn, heads, kv_heads, head_dim, rows, window, apart):
    """`apart`: how many entries the step's keys and values lie behind 16 bytes, and the workspace behind 8."""
    gen = torch.Generator().manual_seed(heads + head_dim + rows)
    dtype, freqs = torch.bfloat16, plain.rope_frequencies(head_dim, 500000.0)
    for at in range(0, len(EDGES), rows):
        lengths = (EDGES[at : at + rows] + EDGES)[:rows]
        kc, vc, table, slots, dense = paged_cache(lengths, kv_heads, head_dim, dtype, at)
        q, k, v = (torch.randn(rows, n * head_dim + 8, generator=gen).to(dtype) for n in (heads, kv_heads, kv_heads))
        angle = torch.tensor([n - 1 for n in lengths], dtype=torch.float64)[:, None] * freqs
        cs = torch.stack([torch.cos(angle), torch.sin(angle)], -1).float().to(DEV)
        c, s = cs[:, None, :, 0].double().cpu(), cs[:, None, :, 1].double().cpu()

        def turned(x, n):
            y = x[:, : n * head_dim].double().view(rows, n, 2, head_dim // 2)
            return torch.cat([y[:, :, 0] * c - y[:, :, 1] * s, y[:, :, 0] * s + y[:, :, 1] * c], -1).to(dtype).double()

        qd, kd, vd = (torch.zeros(rows, t.shape[1] + 8, dtype=dtype, device=DEV) for t in (q, k, v))
        qd[:, : q.shape[1]], kd[:, apart : apart + k.shape[1]], vd[:, apart : apart + v.shape[1]] = q.to(DEV), k.to(DEV), v.to(DEV)
        out = torch.empty(rows, heads * head_dim, dtype=dtype, device=DEV)
        need = kn.attention_workspace(dtype, rows, heads, kv_heads, head_dim, BS, True, max(lengths))
        ws = torch.empty(need + 2, dtype=torch.float32, device=DEV)[apart:]
        for b, n in enumerate(lengths):  # the new position's place holds nothing yet, those behind it never did
            blk = table[slots[b], (n - 1) // BS].long()
            kc[blk, :, (n - 1) % BS :], vc[blk, :, :, (n - 1) % BS :] = float("inf"), float("nan")
        kn.attention(qd, out, heads, kv_heads, head_dim, i32([n - 1 for n in lengths]), i32(range(rows)), i32(slots),
                     i32(range(rows + 1)), table, kc, vc, BS, 1.0 / math.sqrt(head_dim), window, decode=True, max_len=max(lengths),
                     workspace=ws, k_new=kd[:, apart:], v_new=vd[:, apart:], cos_sin=cs)
        qt, kt = turned(q, heads), turned(k, kv_heads)
        for b, n in enumerate(lengths):
            keys, values = (t.double().clone() for t in dense[b])
            keys[n - 1], values[n - 1] = kt[b], v[b, : kv_heads * head_dim].double().view(kv_heads, head_dim)
            full = torch.zeros(n, heads, head_dim, dtype=torch.float64)
            full[n - 1] = qt[b]
            want = plain.attention(full, keys, values, window=window, rows=[n - 1])[n - 1]
            # (the result and the probabilities are rounded to 8 bits, 2^-9 each at most, as in the other tests of this kernel)
            assert rel_err(out[b].view(heads, head_dim), want) < 1.2e-2, (b, n)
            blk, off = table[slots[b], (n - 1) // BS].long(), (n - 1) % BS
            assert torch.equal(vc[blk, :, :, off].cpu(), v[b, : kv_heads * head_dim].view(kv_heads, head_dim))
            assert rel_err(kc[blk, :, off], kt[b]) < 4e-3
        assert int(kn.tickets(torch.device("cuda", torch.cuda.current_device())).abs().max()) == 0


@pytest.mark.parametrize("kv_heads,head_dim", [(64, 64), (64, 128)])
def test_rows_of_more_blocks_than_a_wavefront_has_lanes(kn, kv_heads, head_dim):
    """Whole rows (as many as compute units) of 64 blocks and one or two more or less, whose numbers are read 64 at a time."""
    lengths = [63 * BS, 64 * BS + 1, 65 * BS + 1, 129 * BS]
    got, want = run_attention(kn, None, lengths, [1] * 4, kv_heads, kv_heads, head_dim, torch.bfloat16, 71, decode=True)
    for b, n in enumerate(lengths):
        assert rel_err(got[b], want[b]) < 1.2e-2, n


@pytest.mark.parametrize("rows,kv_heads,head_dim,start", [(17, 8, 128, 12), (21, 8, 64, 16), (3, 64, 64, 32), (3, 64, 128, 80), (33, 8, 192, 14),
                                                          (5, 64, 128, 14), (6, 64, 128, 28), (6, 64, 64, 28), (12, 32, 256, 28),
                                                          (3, 64, 96, 20), (5, 64, 192, 10), (9, 64, 96, 10), (9, 64, 128, 18), (9, 64, 192, 18),
                                                          (9, 64, 64, 18), (10, 64, 64, 48), (18, 64, 96, 14), (5, 64, 64, 28)])
@pytest.mark.parametrize("window", [0, 1000])
def test_long_rows_of_launches_that_fill_the_chip(kn, rows, kv_heads, head_dim, start, window):
    """Launches of half to five times as many rows and kv heads as compute units: rows of up to `start` blocks stay whole, longer ones go
    in shares, which its last workgroup adds up, so that the units have equal parts.  Rows at that line, far beyond it and of one
    key; twice the same, with the counters at zero after each."""
    lengths = ([start * BS, (start - 1) * BS, (start - 1) * BS + 1, 3 * start * BS + 65, 1, start * BS + 1] * rows)[:rows]
    if rows > 6:
        lengths[6:] = [n if n < 200 else 200 + 7 * r for r, n in enumerate(lengths[6:])]
    assert kn.attention_workspace(torch.bfloat16, rows, kv_heads, kv_heads, head_dim, BS, True, max(lengths)) > 0
    outs = []
    for _ in range(2):
        got, want = run_attention(kn, None, lengths, [1] * rows, kv_heads, kv_heads, head_dim, torch.bfloat16, 83, window=window, decode=True)
        for b, n in enumerate(lengths):
            assert rel_err(got[b], want[b]) < 1.2e-2, (b, n)
        assert int(kn.tickets(torch.device("cuda", torch.cuda.current_device())).abs().max()) == 0
        outs.append(got)
    assert torch.equal(*outs)


@pytest.mark.parametrize("rows,heads,kv_heads,head_dim", [(7, 64, 64, 64), (16, 128, 64, 64), (11, 64, 64, 128), (21, 64, 32, 128), (24, 32, 32, 64)])
@pytest.mark.parametrize("window", [0, 70])
def test_rows_of_which_a_unit_holds_more(kn, rows, heads, kv_heads, head_dim, window):
    """Where one block goes at a time at head size 64, and three workgroups are held of 128: rows of every edge of a block and of more blocks than
    a wavefront has lanes."""
    lengths = (EDGES + [64 * BS + 1, 65 * BS, 66 * BS + 1, 3, 70, 190, 500, 700])[-rows:]
    got, want = run_attention(kn, None, lengths, [1] * rows, heads, kv_heads, head_dim, torch.bfloat16, 29, window=window, decode=True)
    for b, n in enumerate(lengths):
        assert rel_err(got[b], want[b]) < 1.2e-2, n


@pytest.mark.parametrize("kv_heads,head_dim", [(8, 128), (2, 192), (1, 256), (8, 64)])
@pytest.mark.parametrize("rows", [1, 3])
def test_bits_do_not_depend_on_the_bound_within_its_bucket(kn, kv_heads, head_dim, rows):
    """A step run directly gives its longest sequence as the bound, a captured one the bound rounded up: the same bits, whatever the
    length; and without a workspace, which up to 256 keys a launch does not need, the same result but for the order of its sums."""
    for n in (64, 150, 193, 230, 256, 257, 700):
        outs = [run_attention(kn, None, [n] * rows, [1] * rows, 2 * kv_heads, kv_heads, head_dim, torch.bfloat16, 91, decode=True, max_len=bound)
                for bound in (n, kn.decode_length_bound(n))]
        assert torch.equal(outs[0][0], outs[1][0]), n
        assert rel_err(*outs[0]) < 8e-3
    lengths = [256, 200, 64][:rows]
    kc, vc, table, slots, dense = paged_cache(lengths, kv_heads, head_dim, torch.bfloat16, 5)
    q = torch.randn(rows, kv_heads * head_dim, generator=torch.Generator().manual_seed(7)).bfloat16().to(DEV)
    out = torch.empty_like(q)
    kn.attention(q, out, kv_heads, kv_heads, head_dim, i32([n - 1 for n in lengths]), i32(range(rows)), i32(slots), i32(range(rows + 1)), table,
                 kc, vc, BS, 1.0 / math.sqrt(head_dim), decode=True, max_len=256)
    for b, n in enumerate(lengths):
        full = torch.zeros(n, kv_heads, head_dim, dtype=torch.float64)
        full[n - 1] = q[b].double().cpu().view(kv_heads, head_dim)
        assert rel_err(out[b].view(kv_heads, head_dim), plain.attention(full, *dense[b], rows=[n - 1])[n - 1]) < 1.2e-2
