"""Prompts through the 32 x 32 score tiles of the windowed attention (`cu_rows` given), and steps of single tokens through
their own kernel, against the general kernel, one wavefront a row and head, at the sizes where tiles, blocks, halves and
shares of the keys end."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PLAIN = dict(sink=False)
CASES = [  # heads, key heads, key size, value size, (new, held) of every sequence, options
    (16, 4, 128, 128, [(1, 0), (32, 0), (33, 63), (2, 64)], dict(window=1024, keep_first=4)),
    (16, 4, 128, 128, [(200, 0), (31, 1000)], dict(window=100, keep_first=70)),
    (8, 2, 128, 128, [(129, 30)], dict(PLAIN, chunk=48)),
    (8, 2, 128, 128, [(70, 90)], dict(PLAIN, window=33)),
    (4, 4, 64, 64, [(127, 0), (130, 1)], PLAIN),
    (6, 3, 64, 48, [(65, 0), (63, 0), (1, 200)], dict(sinks=True)),
    (3, 1, 40, 24, [(97, 31)], PLAIN),
    (8, 2, 112, 80, [(40, 61)], dict(window=64, gate=True)),
    (8, 4, 128, 256, [(77, 51), (3, 0)], dict(PLAIN, maps=2, window=90)),
    (4, 1, 96, 136, [(65, 0)], dict(PLAIN, wide=True)),
    (16, 1, 256, 192, [(33, 31), (64, 0)], PLAIN),
    (4, 1, 200, 104, [(50, 15)], PLAIN),
    (8, 2, 128, 128, [(90, 300)], dict(sinks=True, cap=30.0, log=True, window=200)),
    (8, 2, 64, 64, [(90, 300)], dict(PLAIN, cap=5.0, dist=100, temp=True, wide=True)),
    (8, 2, 128, 128, [(130, 300), (40, 0)], dict(sinks="lowest", window=100)),
    (4, 1, 64, 64, [(200, 30)], dict(sinks="none", chunk=50)), (8, 4, 200, 104, [(100, 90)], dict(sinks="lowest", window=40)),
    (6, 3, 128, 256, [(140, 64)], dict(sinks="none", window=33, keep_first=3)),
    (8, 2, 128, 128, [(130, 300), (40, 0)], dict(sinks="highest", window=100)), (8, 4, 200, 104, [(100, 90)], dict(sinks="highest", window=40)),
]


LENGTHS = [1, 63, 64, 65, 255, 256, 257, 300, 700, 1030]
SINGLE = [  # heads, key heads, key size, value size, options
    (16, 4, 128, 128, dict(window=256, keep_first=70)), (16, 4, 128, 128, dict(PLAIN, chunk=100)),
    (16, 1, 256, 192, PLAIN), (40, 2, 64, 40, dict(sinks=True, gate=True)), (4, 1, 256, 256, PLAIN),
    (8, 4, 128, 256, dict(PLAIN, maps=2, window=600)), (3, 3, 40, 24, dict(window=1, wide=True)),
    (8, 2, 128, 128, dict(sinks=True, cap=30.0, log=True, window=200)),
    (8, 2, 64, 64, dict(PLAIN, cap=5.0, dist=100, temp=True, wide=True)),
    (8, 2, 128, 128, dict(sinks="highest", window=300)),
    (8, 2, 128, 128, dict(sinks="lowest", window=100)), (4, 1, 64, 64, dict(sinks="none", chunk=50))]


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("H,G,D,P,options", SINGLE)
def test_single_tokens(H, G, D, P, options, shared):
    check(H, G, D, P, [(1, n - 1) for n in LENGTHS], options, shared)


@pytest.mark.parametrize("lengths", [[1], [64, 65], [129], [700], [192, 193, 321], [4097], [256, 257, 384, 385, 448, 449]])
@pytest.mark.parametrize("H,G,D,P,options", [(16, 1, 256, 192, PLAIN), (20, 1, 64, 40, dict(sinks=True, gate=True)), (3, 1, 128, 256, PLAIN),
                                             (8, 2, 128, 128, dict(PLAIN, cap=5.0, dist=100, wide=True)),
                                             (24, 1, 40, 72, dict(window=300, keep_first=130)), (64, 8, 64, 64, dict(sinks=True, window=128)),
                                             (16, 8, 64, 64, PLAIN)])
def test_single_tokens_of_few_rows(H, G, D, P, options, lengths):
    """A key head's query heads in several workgroups, down to two heads each, and shares of one block upwards."""
    check(H, G, D, P, [(1, n - 1) for n in lengths], options, True)


@pytest.mark.parametrize("H,G,D,P,options", [(8, 8, 64, 64, dict(sinks=True, window=128)), (128, 64, 64, 40, dict(PLAIN, window=4200, keep_first=300)),
                                             (64, 64, 128, 128, dict(sinks=True, gate=True)), (256, 8, 128, 256, dict(PLAIN, chunk=5000))])
def test_single_tokens_of_more_blocks_than_a_wavefront_has_lanes(H, G, D, P, options):
    """Whole rows (as many tiles of heads as compute units) of 64 blocks and more, whose numbers are read 64 at a time, and rows of an odd
    number of blocks where two go together."""
    check(H, G, D, P, [(1, n - 1) for n in (160, 63 * 64, 64 * 64 + 1, 65 * 64 + 1)], options, True)


@pytest.mark.parametrize("H,G,D,P,rows,start", [(128, 64, 64, 64, 3, 32), (128, 64, 64, 40, 5, 28), (132, 33, 128, 128, 4, 8), (264, 66, 128, 128, 4, 14),
                                                (160, 80, 128, 256, 4, 6), (380, 95, 128, 128, 4, 28), (64, 16, 256, 192, 9, 4), (640, 32, 64, 64, 4, 28)])
@pytest.mark.parametrize("options", [PLAIN, dict(sinks=True, window=700, gate=True)])
def test_single_tokens_of_launches_that_fill_the_chip(H, G, D, P, rows, start, options):
    """Half to twice as many rows and tiles of heads as compute units: rows of up to some `start` blocks stay whole, longer ones go in shares.  Rows
    at that line, far beyond it and of one key."""
    check(H, G, D, P, [(1, n - 1) for n in [start * 64, (start - 1) * 64, start * 64 + 1, 1, 2 * start * 64 + 65, 3, 70, 130, 260][:rows]], options, True)


@pytest.mark.parametrize("H,G,D,P,seqs,options", CASES)
def test_tiles_of_32_rows(H, G, D, P, seqs, options):
    check(H, G, D, P, seqs, options, False)


def check(H, G, D, P, seqs, options, shared):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(H * 1000 + D + P)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    o = dict(options)
    maps = o.pop("maps", 1)
    blocks = [-(-(n + held) // 64) for n, held in seqs]
    order = torch.randperm(sum(blocks), generator=gen).int()
    table = torch.zeros(len(seqs), max(blocks), dtype=torch.int32)
    at = 0
    for b, n in enumerate(blocks):
        table[b, :n] = order[at : at + n]
        at += n
    k = rand(sum(blocks), G // maps, 64, maps * D).bfloat16()
    v = rand(sum(blocks), G // maps, P, 64).bfloat16()
    for b, (n, held) in enumerate(seqs):  # what was never written may be anything
        if (n + held) % 64:
            v[table[b, blocks[b] - 1].long(), :, :, (n + held) % 64 :] = float("nan")
            k[table[b, blocks[b] - 1].long(), :, (n + held) % 64 :] = float("inf")
    rows = sum(n for n, _ in seqs)
    q = rand(rows, H * D).bfloat16()
    more = dict(window=o.get("window", 0), keep_first=o.get("keep_first", 0), sink=o.get("sink", True), maps=maps,
                chunk=o.get("chunk", 0), softcap=o.get("cap", 0.0))
    if "sinks" in o:
        more["sink_values"] = rand(H)
        most = torch.finfo(torch.float32).max
        odd = {"none": [float("-inf")], "lowest": [-most, -2.4e38, -2.0e38, float("-inf")], "highest": [most, 2.4e38, 2.0e38]}.get(o["sinks"], [])
        for i in range(H if odd else 0):  # (a sink that says no more than an absent one, or all there is, beside ordinary ones)
            if i % 3 < 2:
                more["sink_values"][i] = odd[i % len(odd)]
    if "gate" in o:
        more["gate"] = rand(rows, H).bfloat16()
    if "wide" in o:
        more["wide_gate"] = rand(rows, H * P)
    if "temp" in o:
        more["temp"] = 1 + 0.1 * rand(H)
    if "log" in o:
        more["log_bias"] = (rand(H).abs(), rand(H).abs())
    if "dist" in o:
        more["distance_bias"] = rand(H, o["dist"])
    pos = i32(held + i for n, held in seqs for i in range(n))
    seq = i32(b for b, (n, _) in enumerate(seqs) for _ in range(n))
    starts = i32([sum(n for n, _ in seqs[:b]) for b in range(len(seqs) + 1)])
    kn = HipKernels()
    for dtype in (torch.float32, torch.bfloat16):
        got, want = (torch.full((rows, H * P), float("nan"), dtype=dtype, device="cuda") for _ in range(2))
        args = (H, G, D, P, pos, seq, i32(range(len(seqs))), table.cuda(), k, v, 64, D ** -0.5)
        how = dict(cu_rows=starts)
        if rows == len(seqs):
            how = dict(decode=True)
            longest = max(n + held for n, held in seqs)
            need = kn.sink_attention_workspace(torch.bfloat16, rows, rows, H, G, D, P, 64, more["window"], more["keep_first"],
                                               longest, chunk=more["chunk"])
            if shared and need:
                how.update(max_len=longest, workspace=torch.full((need,), float("nan"), device="cuda"))
        for _ in range(2):  # (a launch leaves the tickets as it found them)
            got.fill_(float("nan"))
            kn.sink_attention(q, got, *args, **how, **more)
        # rows of q 4 entries more than a multiple of 8 apart, and starting on 8 bytes: the same kernel, the same bits
        wide = torch.zeros(rows, H * D + (4 if H * D % 8 == 0 else 0) + 8, dtype=q.dtype, device="cuda")
        wide[:, 4 : 4 + H * D] = q
        apart = torch.full_like(got, float("nan"))
        kn.sink_attention(wide[:, 4 : 4 + H * D], apart, *args, **how, **more)
        assert torch.equal(apart, got)
        if "workspace" in how:  # the shares added up by their last workgroup, or by a second launch: the same bits
            counters = torch.zeros(1024, dtype=torch.int32, device="cuda")
            for _ in range(2):  # (a launch leaves the counters as it found them)
                apart.fill_(float("nan"))
                kn.sink_attention(q, apart, *args, **how, **more, tickets=counters)
                assert torch.equal(apart, got) and not counters.any()
            assert not kn.tickets(q.device).any()  # (the object's own are for the causal attention)
        kn.force_generic = True
        kn.sink_attention(q, want, *args, **more)
        kn.force_generic = False
        # Sums of N terms in another order differ by at most 2 N 2^-24 of sum p |v| <= max |v|, the exponentials'
        # arguments (up to 30 with the log bias) by 2^-22 of themselves: 1.4e-4 + 1e-5 of 4.7 at N = 1 031, and what
        # is seen is a hundredth of that.  In bfloat16 the two may round to neighbours: 2^-8 of the value.
        assert torch.isfinite(want).all()
        far = (got.float() - want.float()).abs()
        assert (far <= 7e-5 + (want.float().abs() * 2 ** -7 if dtype == torch.bfloat16 else 0)).all(), far.max()


def test_scratch_of_very_many_rows_and_heads():
    """2^32 rows and key heads together are no number of 32 bits; so many share nothing out and ask for no scratch."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    ask = HipKernels().sink_attention_workspace
    assert ask(torch.bfloat16, 1 << 17, 1 << 17, 1 << 15, 1 << 15, 64, 64, 64, 0, 0, 4096) == 0
    assert ask(torch.bfloat16, 2, 2, 16, 4, 64, 64, 64, 0, 0, 4096) > 0


@pytest.mark.parametrize("H,G,D,P,options", [(8, 2, 128, 128, PLAIN), (4, 1, 64, 64, dict(PLAIN, window=70)), (2, 2, 200, 104, PLAIN)])
def test_a_row_has_the_same_bits_whatever_its_neighbours(H, G, D, P, options):
    """A prompt's row beside rows of ordinary scores, beside rows of scores 60 times as large (whose maximum moves in every
    block), and in a portion of its own length."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(D)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    held, rows = 150, 100
    k, v, q = rand(4, G, 64, D).bfloat16(), rand(4, G, P, 64).bfloat16(), 3 * rand(rows, H * D)
    kn = HipKernels()

    def run(first, q):
        n = q.shape[0]
        out = torch.full((n, H * P), float("nan"), device="cuda")
        kn.sink_attention(q.bfloat16(), out, H, G, D, P, i32(range(held + first, held + first + n)), i32([0] * n), i32([0]),
                          i32([2, 0, 3, 1]).view(1, 4), k, v, 64, D ** -0.5, cu_rows=i32([0, n]), **options)
        return out

    want = run(0, q)
    pushed = q.clone()
    pushed[1::2] *= 60
    assert torch.equal(run(0, pushed)[::2], want[::2])
    for first, n in ((0, 2), (31, 40), (57, 43)):
        assert torch.equal(run(first, q[first : first + n]), want[first : first + n]), (first, n)
