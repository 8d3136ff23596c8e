"""The state-space scan in chunks of 64 tokens against the walk token by token (no scratch given), at the sizes where
chunks, blocks of 16 tokens, slices of columns and halves of channels end."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,H,G,N,P,given,shift", [
    ([128], 4, 2, 128, 64, False, 0.0), ([1, 129, 63, 64, 65], 4, 1, 128, 64, False, 0.0), ([150], 2, 2, 30, 17, False, 0.0),
    ([140, 16], 3, 3, 48, 40, False, 0.0), ([130], 2, 1, 256, 100, False, 0.0), ([200], 2, 2, 132, 64, False, 0.0),
    ([130, 70], 2, 2, 256, 129, True, 0.0), ([128], 1, 1, 64, 65, True, 0.0), ([129], 2, 2, 30, 18, True, 0.0),
    ([131], 2, 1, 128, 64, False, 8.0), ([131], 2, 1, 128, 64, False, -8.0), ([128] + [1] * 70, 2, 1, 64, 32, False, 0.0)])
def test_chunks_of_the_state_space_scan(lens, H, G, N, P, given, shift):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(N * P + len(lens))
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    rows, batch = sum(lens), len(lens)
    x, b, c, dt = rand(rows, H * (P - given)), 0.3 * rand(rows, G * N), 0.3 * rand(rows, G * N), rand(rows, H)
    made = (rand(H) - 3.0 + shift, 0.5 * rand(H) + 1.0, rand(H))
    more = {}
    if given:  # a matrix memory's: decays and steps as they are, and a column of ones
        made, dt, more = (None, None, None), dt.abs(), dict(decay=torch.sigmoid(rand(rows, H) + 3.0), ones=True)
    state = rand(batch, H, P, N)
    cu = i32(sum(lens[:i]) for i in range(batch + 1))
    kn = HipKernels()
    need = kn.ssd_scan_workspace(batch, H, P, N, max(lens), rows)
    assert need > 0 and kn.ssd_scan_workspace(batch, H, P, N, 1, batch) == 0
    got = {}
    for scratch in (None, torch.full((need,), float("nan"), device="cuda")):
        y, end = torch.full((rows, H * P), float("nan"), device="cuda"), state.clone()
        how = {} if scratch is None else dict(max_rows=max(lens), workspace=scratch, chunks=True)
        kn.ssd_scan(x, b, c, dt, *made, end, y, H, P, N, G, i32(reversed(range(batch))), cu, batch, **how, **more)
        got[scratch is not None] = y, end
    # Sums of up to 200 tokens' terms and then N channels' in another order: at most (3 x 200 + N) roundings of 2^-24 at
    # the size of the terms' absolute sum, which the largest state entry times sum_n |C_n| bounds.
    (walked, end0), (chunked, end1) = got[False], got[True]
    assert torch.isfinite(walked).all() and torch.isfinite(end0).all()
    unit = (3 * 200 + N) * 2.0 ** -24 * end0.abs().max().clamp(min=float(state.abs().max()))
    assert (end0 - end1).abs().max() <= unit
    assert (walked - chunked).abs().max() <= unit * c.abs().view(rows, G, N).sum(-1).max() + 1e-6 * walked.abs().max()


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("what", ["x", "b", "c", "dt"])
@pytest.mark.parametrize("at", [0, 21, 47, 63, 64, 110])
def test_what_is_no_number_reaches_later_tokens_only(what, at, given):
    """A NaN or an infinity at a token: the results before it stay what they are without it, in chunks as token by token,
    and from it on the same ones are no numbers."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(at)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    rows, H, G, N, P = 140, 2, 1, 64, 48
    plain = dict(x=rand(rows, H * (P - given)), b=0.3 * rand(rows, G * N), c=0.3 * rand(rows, G * N), dt=rand(rows, H).abs())
    made = (rand(H) - 3.0, 0.5 * rand(H) + 1.0, rand(H))
    more = {}
    if given:
        made, more = (None, None, None), dict(decay=torch.sigmoid(rand(rows, H) + 3.0), ones=True)
    state = rand(1, H, P, N)
    kn = HipKernels()
    need = kn.ssd_scan_workspace(1, H, P, N, rows, rows)
    got = {}
    for case, bad in (("plain", None), ("nan", float("nan")), ("inf", float("inf"))):
        t = {name: x.clone() for name, x in plain.items()}
        if bad is not None:
            t[what][at, :1] = bad
        for scratch in (None, torch.full((need,), float("nan"), device="cuda")):
            y, end = torch.full((rows, H * P), float("nan"), device="cuda"), state.clone()
            how = {} if scratch is None else dict(max_rows=rows, workspace=scratch, chunks=True)
            kn.ssd_scan(t["x"], t["b"], t["c"], t["dt"], *made, end, y, H, P, N, G, i32([0]), i32([0, rows]), 1, **how, **more)
            got[case, scratch is not None] = y, end
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
    x, b, c, dt = rand(rows, H * P), 0.3 * rand(rows, G * N), 0.3 * rand(rows, G * N), rand(rows, H)
    made, state = (rand(H) - 3.0, 0.5 * rand(H) + 1.0, rand(H)), rand(batch, H, P, N)
    kn = HipKernels()
    need = kn.ssd_scan_workspace(batch, H, P, N, max(lens), rows)
    a_chunk = need // (rows // 64 + batch)
    got = []
    for floats in (need, chunks * a_chunk):
        y, end = torch.full((rows, H * P), float("nan"), device="cuda"), state.clone()
        kn.ssd_scan(x, b, c, dt, *made, end, y, H, P, N, G, i32(range(batch)), i32(sum(lens[:i]) for i in range(batch + 1)),
                    batch, max_rows=max(lens), workspace=torch.full((floats,), float("nan"), device="cuda"), chunks=True)
        got.append((y, end))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_scratch_is_bounded():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    for rows, batch, heads, P, N in ((65536, 1, 32, 64, 128), (16384, 8, 4, 513, 256), (1 << 20, 4, 128, 64, 128)):
        assert 0 < kn.ssd_scan_workspace(batch, heads, P, N, rows // batch, rows) <= 64 << 20


def test_short_sequences_beside_a_long_one_are_walked():
    """More chunks than the chip takes at once: sequences of fewer than 48 tokens have the bits of the walk token by token,
    the others those of a launch of their own in chunks."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    gen = torch.Generator().manual_seed(48)
    rand = lambda *s: torch.randn(*s, generator=gen).cuda()
    i32 = lambda v: torch.tensor(list(v), dtype=torch.int32, device="cuda")
    lens = [1, 47, 200, 48, 64, 130] + [2] * 40 + [49]
    rows, batch, H, G, N, P = sum(lens), len(lens), 8, 4, 64, 48
    x, b, c, dt = rand(rows, H * P), 0.3 * rand(rows, G * N), 0.3 * rand(rows, G * N), rand(rows, H)
    made, state = (rand(H) - 3.0, 0.5 * rand(H) + 1.0, rand(H)), rand(batch, H, P, N)
    kn = HipKernels()
    need = lambda mine: kn.ssd_scan_workspace(len(mine), H, P, N, max(mine), sum(mine)) if max(mine) >= 128 else 0

    def run(first, mine, floats):
        n, at, B = sum(mine), sum(lens[:first]), len(mine)
        y, end = torch.full((n, H * P), float("nan"), device="cuda"), state[first : first + B].clone()
        part = lambda t: t[at : at + n]
        how = dict(max_rows=max(mine), min_rows=min(mine), workspace=torch.full((floats,), float("nan"), device="cuda"), chunks=True) if floats else {}
        kn.ssd_scan(part(x), part(b), part(c), part(dt), *made, end, y, H, P, N, G, i32(range(B)),
                    i32(sum(mine[:i]) for i in range(B + 1)), B, **how)
        return y, end

    (got, got_end), (walked, walked_end) = run(0, lens, need(lens)), run(0, lens, 0)
    unit = (3 * 200 + N) * 2.0 ** -24 * walked_end.abs().max().clamp(min=float(state.abs().max()))  # (as above)
    for s, n in enumerate(lens):
        at = sum(lens[:s])
        if n < 48:
            assert torch.equal(got[at : at + n], walked[at : at + n]) and torch.equal(got_end[s], walked_end[s])
        else:
            assert (got[at : at + n] - walked[at : at + n]).abs().max() <= unit * c.abs().view(rows, G, N).sum(-1).max() + 1e-6 * walked.abs().max()
            if need([n]):  # (a launch of its own is in chunks too)
                alone, end = run(s, [n], need([n]))
                assert torch.equal(got[at : at + n], alone) and torch.equal(got_end[s], end[0])


def test_which_launches_are_faster_in_chunks():
    """Sizes far from where both ways take as long: few long sequences in chunks, very many or short ones of small states
    token by token."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    ask = HipKernels().ssd_scan_in_chunks
    assert ask(1, 32, 64, 128, 2048, 2048) and ask(8, 32, 64, 128, 512, 4096) and ask(1, 4, 513, 256, 2048, 2048)
    assert ask(71, 32, 64, 128, 2000, 2070)
    assert not ask(1, 32, 64, 128, 100, 100) and not ask(64, 32, 64, 128, 1, 64) and not ask(8, 32, 16, 64, 1000, 8000)
    assert not ask(32, 32, 64, 16, 256, 32 * 256) and not ask(1, 32, 64, 300, 2048, 2048)
