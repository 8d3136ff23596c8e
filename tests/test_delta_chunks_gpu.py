"""The gated delta rule in chunks of 64 tokens against the walk token by token (no scratch given), at the sizes where
chunks, blocks of 16 tokens, value slices and rows of key channels end."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,H,G,N,P,channel,shift", [
    ([64], 2, 1, 128, 128, True, 0.0), ([1, 65, 16], 4, 2, 128, 128, False, 0.0), ([129, 63], 3, 3, 128, 128, True, 0.0),
    ([200], 2, 2, 48, 40, True, 0.0), ([80, 17, 128], 2, 1, 64, 256, False, 0.0), ([70], 2, 1, 30, 17, True, 0.0),
    ([66], 1, 1, 16, 16, False, 0.0), ([130], 2, 1, 128, 32, True, 8.0), ([130], 2, 1, 128, 32, False, 8.0),
    ([130], 2, 1, 128, 32, True, -8.0), ([57] + [1] * 70, 2, 1, 64, 32, True, 0.0)])
def test_chunks_of_the_delta_rule(lens, H, G, N, P, channel, shift):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(N * P + len(lens))
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    rows, batch = sum(lens), len(lens)
    q, k, v, beta = rand(rows, G * N), rand(rows, G * N), rand(rows, H * P), rand(rows, H)
    k[1::3] = 0.9 * k[0::3][: k[1::3].shape[0]] + 0.1 * k[1::3]  # keys that overwrite one another
    n_decay = H * N if channel else H
    a, dt_bias, a_log = 0.3 * rand(rows, n_decay), rand(n_decay) - 3.0 + shift, 0.5 * rand(H) + 1.0
    state = rand(batch, H, P, N)
    cu = i32(sum(lens[:b]) for b in range(batch + 1))
    kn = HipKernels()
    need = kn.delta_scan_workspace(rows, batch, H, N, P, max(lens))
    assert need > 0 and kn.delta_scan_workspace(batch, batch, H, N, P, 1) == 0
    got = {}
    for scratch in (None, torch.full((need,), float("nan"), device="cuda")):
        out, end, qq, kk = torch.full((rows, H * P), float("nan"), device="cuda"), state.clone(), q.clone(), k.clone()
        more = {} if scratch is None else dict(max_rows=max(lens), workspace=scratch)
        kn.delta_scan(qq, kk, v, beta, a, dt_bias, a_log, end, out, H, G, N, P, N ** -0.5, 1e-6,
                      i32(reversed(range(batch))), cu, batch, channel_decay=channel, **more)
        got[scratch is not None] = out, end
    for walked, chunked in zip(got[False], got[True]):
        # Every step is a contraction, so an error made at a token is not enlarged by the later ones: at most some 4
        # roundings of 2^-24 a token at the result's size, 200 tokens.
        assert torch.isfinite(walked).all()
        assert (walked - chunked).abs().max() <= 200 * 4 * 2.0 ** -24 * walked.abs().max()


@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "a"])
@pytest.mark.parametrize("at", [0, 21, 47, 63, 64, 90])
def test_what_is_no_number_reaches_later_tokens_only(what, at, channel):
    """A NaN or an infinity at a token: the results before it stay what they are without it, in chunks as token by token,
    and from it on the same ones are no numbers."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(at)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    rows, H, G, N, P = 100, 2, 1, 64, 48
    given = dict(q=rand(rows, G * N), k=rand(rows, G * N), v=rand(rows, H * P), beta=rand(rows, H),
                 a=0.3 * rand(rows, H * N if channel else H))
    dt_bias, a_log, state = rand(given["a"].shape[1]) - 3.0, 0.5 * rand(H) + 1.0, rand(1, H, P, N)
    kn = HipKernels()
    need = kn.delta_scan_workspace(rows, 1, H, N, P, rows)
    got = {}
    for case, bad in (("plain", None), ("nan", float("nan")), ("inf", float("inf"))):
        t = {name: x.clone() for name, x in given.items()}
        if bad is not None:
            t[what][at, :1] = bad
        for scratch in (None, torch.full((need,), float("nan"), device="cuda")):
            out, end = torch.full((rows, H * P), float("nan"), device="cuda"), state.clone()
            more = {} if scratch is None else dict(max_rows=rows, workspace=scratch)
            kn.delta_scan(t["q"].clone(), t["k"].clone(), t["v"], t["beta"], t["a"], dt_bias, a_log, end, out, H, G, N, P,
                          N ** -0.5, 1e-6, i32([0]), i32([0, rows]), 1, channel_decay=channel, **more)
            got[case, scratch is not None] = out, end
    for bad in ("nan", "inf"):
        (walked, end0), (chunked, end1) = got[bad, False], got[bad, True]
        assert torch.equal(chunked[:at], got["plain", True][0][:at])
        assert torch.equal(torch.isfinite(walked), torch.isfinite(chunked))
        assert torch.equal(torch.isfinite(end0), torch.isfinite(end1))


@pytest.mark.parametrize("lens", [[300], [65, 1, 130, 64, 70]])
@pytest.mark.parametrize("chunks", [1, 2, 3])
def test_rounds_of_chunks_make_the_same_bits(lens, chunks):
    """A workspace of fewer chunks than the step has: the chunks go in rounds, from state to state."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(chunks)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    rows, batch, H, G, N, P = sum(lens), len(lens), 4, 2, 64, 80
    q, k, v, beta, a = rand(rows, G * N), rand(rows, G * N), rand(rows, H * P), rand(rows, H), rand(rows, H * N)
    dt_bias, a_log, state = rand(H * N) - 3.0, 0.5 * rand(H) + 1.0, rand(batch, H, P, N)
    kn = HipKernels()
    need = kn.delta_scan_workspace(rows, batch, H, N, P, max(lens))
    a_chunk = need // (rows // 64 + batch)
    got = []
    for floats in (need, chunks * a_chunk):
        out, end = torch.full((rows, H * P), float("nan"), device="cuda"), state.clone()
        kn.delta_scan(q.clone(), k.clone(), v, beta, a, dt_bias, a_log, end, out, H, G, N, P, N ** -0.5, 1e-6, i32(range(batch)),
                      i32(sum(lens[:b]) for b in range(batch + 1)), batch, channel_decay=True, max_rows=max(lens),
                      workspace=torch.full((floats,), float("nan"), device="cuda"))
        got.append((out, end))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("lens", [[64], [65], [128], [129, 191, 64], [70, 320]])
@pytest.mark.parametrize("N,P", [(128, 16), (44, 36), (4, 3)])
def test_the_walk_over_chunks_keeps_to_its_columns(lens, N, P):
    """Values and results that are columns of wider matrices, odd and even numbers of chunks, heads' values that end inside
    a tile of 16 columns: the bits of dense matrices, and nothing beside them is read or written."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(N + P)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    rows, batch, H = sum(lens), len(lens), 3
    q, k, beta, a = rand(rows, H * N), rand(rows, H * N), rand(rows, H), 0.3 * rand(rows, H)
    dt_bias, a_log, state = rand(H) - 3.0, 0.5 * rand(H) + 1.0, rand(batch, H, P, N)
    kn = HipKernels()
    scratch = torch.full((kn.delta_scan_workspace(rows, batch, H, N, P, max(lens)),), float("nan"), device="cuda")
    v, got = rand(rows, H * P), []
    for extra in (0, 5):
        wide = torch.full((rows + 64, H * P + 2 * extra), float("nan"), device="cuda")
        wide[:rows, extra : extra + H * P] = v
        out, end = torch.full_like(wide, 7.0), state.clone()
        cut = lambda m: m[:rows, extra : extra + H * P]
        kn.delta_scan(q.clone(), k.clone(), cut(wide), beta, a, dt_bias, a_log, end, cut(out), H, H, N, P, N ** -0.5, 1e-6,
                      i32(range(batch)), i32(sum(lens[:b]) for b in range(batch + 1)), batch, channel_decay=False,
                      max_rows=max(lens), workspace=scratch)
        got.append((cut(out).clone(), end))
        cut(out).fill_(7.0)
        assert (out == 7.0).all()
    for dense, apart in zip(*got):
        assert torch.isfinite(dense).all() and torch.equal(dense, apart)


def test_scratch_is_bounded():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    for rows, batch, heads in ((65536, 1, 16), (8192, 64, 32), (1 << 20, 4, 128)):
        assert 0 < kn.delta_scan_workspace(rows, batch, heads, 128, 128, rows // batch) <= 64 << 20


@pytest.mark.parametrize("channel,least", [(True, 24), (False, 48)])
def test_short_sequences_beside_a_long_one_are_walked(channel, least):
    """More chunks than the chip takes at once: sequences of fewer than `least` tokens have the bits of the walk token by
    token, the others those of a launch of their own in chunks."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(least)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    lens = [1, least - 1, 100, least, 64] + [2] * 40 + [least + 1]
    rows, batch, H, G, N, P = sum(lens), len(lens), 8, 4, 64, 48
    q, k, v, beta, a = rand(rows, G * N), rand(rows, G * N), rand(rows, H * P), rand(rows, H), rand(rows, H * N if channel else H)
    dt_bias, a_log, state = rand(a.shape[1]) - 3.0, 0.5 * rand(H) + 1.0, rand(batch, H, P, N)
    kn = HipKernels()

    all_lens = lens

    def run(first, lens, floats):
        n, at, B = sum(lens), sum(all_lens[:first]), len(lens)
        out, end = torch.full((n, H * P), float("nan"), device="cuda"), state[first : first + B].clone()
        part = lambda x: x[at : at + n].clone()
        more = dict(max_rows=max(lens), min_rows=min(lens), workspace=torch.full((floats,), float("nan"), device="cuda")) if floats else {}
        kn.delta_scan(part(q), part(k), part(v), part(beta), part(a), dt_bias, a_log, end, out, H, G, N, P, N ** -0.5, 1e-6,
                      i32(range(B)), i32(sum(lens[:b]) for b in range(B + 1)), B, channel_decay=channel, **more)
        return out, end

    need = lambda lens: kn.delta_scan_workspace(sum(lens), len(lens), H, N, P, max(lens))
    (got, got_end), (walked, walked_end) = run(0, lens, need(lens)), run(0, lens, 0)
    for b, n in enumerate(lens):
        at = sum(lens[:b])
        if n < least:
            assert torch.equal(got[at : at + n], walked[at : at + n]) and torch.equal(got_end[b], walked_end[b])
        else:
            far = 64 * 4 * 2.0 ** -24  # (as above: at most some 4 roundings a token, here up to 100 tokens)
            assert (got[at : at + n] - walked[at : at + n]).abs().max() <= 2 * far * walked.abs().max()
            if need([n]):  # (a launch of its own is in chunks too)
                alone, end = run(b, [n], need([n]))
                assert torch.equal(got[at : at + n], alone) and torch.equal(got_end[b], end[0])


def test_which_launches_are_faster_in_chunks():
    """Sizes far from where both ways take as long: few long sequences in chunks, very many or short ones token by token."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    ask = HipKernels().delta_scan_in_chunks
    for channel in (False, True):
        assert ask(256, 1, 16, 128, 128, 256, channel) and ask(8192, 1, 16, 128, 128, 8192, channel) and ask(3990, 70, 16, 128, 128, 2000, channel)
        assert not ask(16, 1, 16, 128, 128, 16, channel) and not ask(256, 256, 16, 128, 128, 1, channel)
        assert not ask(70 * 57, 70, 16, 64, 64, 57, channel)
    assert not ask(70 * 200, 70, 16, 128, 128, 200, False) and ask(70 * 200, 70, 16, 128, 128, 200, True)
