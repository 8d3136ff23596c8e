"""Kernels that take many rows (512 and more) in tiles against the same kernels' paths for fewer rows: a row's sums
are the same whatever tile it lies in, so every result is equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def kn():
    from longbow_quarrel_amd.kernels.hip import HipKernels
    return HipKernels()


def rnd(*shape, seed):
    return torch.empty(shape).normal_(0, 1.0, generator=torch.Generator().manual_seed(seed)).to(DEV)


def i32(values):
    return torch.tensor(list(values), dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("lengths", [(512,), (513, ), (1, 2, 1, 3, 505, 7, 1), (255, 256, 2, 1, 3)])
def test_convolution_of_many_rows(kn, lengths, taps, dtype):
    C, wide = 132, 140
    rows, n = sum(lengths), len(lengths)
    x = rnd(rows, wide, seed=1).to(dtype)[:, 4 : 4 + C]
    w, b = rnd(C, taps, seed=2), rnd(C, seed=3)
    first = rnd(n + 1, taps - 1, C, seed=4)
    start = [0 if s % 2 else 11 for s in range(n)]  # (some go on after earlier tokens)
    slot = [n - s for s in range(n)]

    def run(state, out, lo, hi, at):  # the rows lo .. hi - 1 of every sequence that has them
        live = [s for s in range(n) if lengths[s] > lo]
        take = [min(hi, lengths[s]) - lo for s in live]
        cu = [0]
        for m in take:
            cu.append(cu[-1] + m)
        pick = torch.cat([torch.arange(at[s] + lo, at[s] + lo + m) for s, m in zip(live, take)]).to(DEV)
        xs, one = (x, out) if len(pick) == rows else (x[pick], torch.zeros((len(pick), C), dtype=dtype, device=DEV))
        kn.causal_conv(xs, w, b, state, one, i32(start[s] + lo + r for s, m in zip(live, take) for r in range(m)),
                       i32(i for i, m in enumerate(take) for _ in range(m)), i32(slot[s] for s in live),
                       i32(start[s] + lo for s in live), i32(start[s] + lo + m for s, m in zip(live, take)), i32(cu), len(live))
        if one is not out:
            out[pick] = one

    at = [sum(lengths[:s]) for s in range(n)]
    whole, parts = torch.zeros((rows, C), dtype=dtype, device=DEV), torch.zeros((rows, C), dtype=dtype, device=DEV)
    sw, sp = first.clone(), first.clone()
    run(sw, whole, 0, max(lengths), at)
    for lo in range(0, max(lengths), 97):
        run(sp, parts, lo, lo + 97, at)
    assert torch.equal(whole, parts)
    assert torch.equal(sw, sp)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [512, 514, 1025])
@pytest.mark.parametrize("group,groups,wlen", [(128, 3, 384), (64, 17, 64), (4, 2, 8), (100, 9, 900), (128, 8, 0)])
def test_gated_norms_of_many_rows(kn, group, groups, wlen, rows, dtype):
    n = group * groups
    y, z = rnd(rows, n + 8, seed=5)[:, 4 : 4 + n], rnd(rows, n, seed=6)
    wt = rnd(wlen, seed=7) if wlen else None
    y[5, 0], z[rows - 1, n - 1], y[rows - 2, 0] = float("nan"), float("-inf"), float("inf")
    for gate, before in (("silu", True), ("silu", False), ("sigmoid", False)):
        got, want = torch.zeros((rows, n), dtype=dtype, device=DEV), torch.zeros((rows, n), dtype=dtype, device=DEV)
        kn.gated_rmsnorm(y, z, wt, 1e-5, group, got, gate_first=before, gate=gate)
        for lo in range(0, rows, 300):
            kn.gated_rmsnorm(y[lo : lo + 300], z[lo : lo + 300], wt, 1e-5, group, want[lo : lo + 300], gate_first=before, gate=gate)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(3.0), want.nan_to_num(3.0)), gate


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("group,groups,wlen,rows", [(128, 1, 128, 8193), (64, 3, 64, 4099), (4, 2, 8, 5121), (100, 9, 900, 1140), (128, 16, 0, 513)])
def test_gated_norms_of_many_rows_and_few_groups(kn, group, groups, wlen, rows, dtype):
    """As many rows as a few groups need for four rows a thread."""
    test_gated_norms_of_many_rows(kn, group, groups, wlen, rows, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,pieces", [(1, 4, 1), (3, 260, 0), (3, 260, 5), (70, 1028, 2), (7, 130, 2), (5, 33, 3)])
def test_dynamic_tanh_in_fours(kn, rows, width, pieces, dtype):
    """Widths in fours and others, against 64 bits; x off a multiple of 16 bytes gives the same as on one."""
    x, w, b, alpha = rnd(rows, width, seed=8), rnd(width, seed=9), rnd(width, seed=10), rnd(1, seed=11)
    delta = rnd(pieces, rows, width, seed=12) if pieces else None
    outs = []
    for off in (0, 1):
        held = torch.zeros(rows * width + 1, device=DEV)[off : off + rows * width].view(rows, width)
        held.copy_(x)
        out = torch.zeros((rows, width), dtype=dtype, device=DEV)
        kn.dynamic_tanh(held, w, b, alpha, out, delta=delta, delta_scale=0.5)
        stream = x.double() + (0.5 * delta.double().sum(0) if pieces else 0.0)
        # (a rounding of 2^-24 a term at the stream's size; the tangent's slope is 1, its own error and the weights' two roundings 4 more)
        bound = 2.0 ** -24 * 8 * (pieces + 1) * (1.0 + stream.abs())
        assert ((held.double() - stream).abs() <= bound).all()
        want = torch.tanh(alpha.double() * stream) * w.double() + b.double()
        slack = bound * (1.0 + alpha.abs().double()) * (1.0 + w.abs().double()) + 2.0 ** -21 * (want.abs() + b.abs().double())
        assert ((out.double() - want).abs() <= slack + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)).all()
        outs.append((held.clone(), out))
        if pieces:
            kn.add_scaled(held, delta, -0.5)
            assert ((held.double() - x.double()).abs() <= 2 * bound).all()
    for on, other in zip(*outs):
        assert (on.double() - other.double()).abs().max() <= 2.0 ** -7 * (1.0 + on.double().abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,pieces", [(131073, 4, 1), (521, 1028, 0), (521, 1028, 5), (1030, 516, 2)])
def test_dynamic_tanh_of_many_entries(kn, rows, width, pieces, dtype):
    """As many entries as are taken in fours."""
    test_dynamic_tanh_in_fours(kn, rows, width, pieces, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 130])
@pytest.mark.parametrize("pieces,extra", [(1, False), (2, True), (4, False)])
def test_postnorm_of_every_width(kn, width, pieces, extra, dtype):
    rows = 3
    x, y, w, nw = rnd(rows, width, seed=13), rnd(pieces, rows, width, seed=14), rnd(width, seed=15), rnd(width, seed=16)
    scales = [0.5, -1.0, 2.0, 1.0][:pieces]
    more = rnd(rows, width, seed=17) if extra else None
    h = torch.zeros((rows, width), dtype=dtype, device=DEV)
    held = x.clone()
    kn.postnorm_residual(held, y if pieces > 1 else y[0], scales, w, 1e-5, extra=more, next_weight=nw, next_eps=1e-3, h=h)
    v = sum(s * y[p].double() for p, s in enumerate(scales))
    stream = x.double() + v / (v.square().mean(1, keepdim=True) + 1e-5).sqrt() * w.double() + (more.double() if extra else 0.0)
    # (sums of a row in a tree of at most 8 + 8 + 2 levels, and some ten roundings more, of 2^-24 at the largest entry's size)
    bound = 2.0 ** -24 * 32 * (1.0 + stream.abs().max())
    assert (held.double() - stream).abs().max() <= bound
    want = stream / (stream.square().mean(1, keepdim=True) + 1e-3).sqrt() * nw.double()
    slack = 2 * bound * (1.0 + nw.abs().double().max()) + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
    assert ((h.double() - want).abs() <= slack).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [2052, 3072, 3076, 5120, 5124, 6144, 6148, 8188])
@pytest.mark.parametrize("pieces,extra", [(1, True), (2, False), (3, True), (4, False)])
def test_postnorm_of_many_wide_rows(kn, width, pieces, extra, dtype):
    """As few as ask for everything ahead of the sums and as many as do not: the same bits, and 64 bits' results within the bound above."""
    rows = max(513, 11000000 // (width * (pieces + 1)) + 1)
    x, y, w, nw = rnd(rows, width, seed=13), rnd(pieces, rows, width, seed=14), rnd(width, seed=15), rnd(width, seed=16)
    scales = [0.5, -1.0, 2.0, 1.0][:pieces]
    more = rnd(rows, width, seed=17) if extra else None
    outs = []
    for n in (rows, 3):
        held, h = x[:n].clone(), torch.zeros((n, width), dtype=dtype, device=DEV)
        part = y[:, :n].contiguous()
        kn.postnorm_residual(held, part if pieces > 1 else part[0], scales, w, 1e-5, extra=more[:n] if extra else None, next_weight=nw,
                             next_eps=1e-3, h=h)
        outs.append((held, h))
    for a, b in zip(*outs):
        assert torch.equal(a[:3], b)
    v = sum(s * y[p].double() for p, s in enumerate(scales))
    stream = x.double() + v / (v.square().mean(1, keepdim=True) + 1e-5).sqrt() * w.double() + (more.double() if extra else 0.0)
    assert (outs[0][0].double() - stream).abs().max() <= 2.0 ** -24 * 32 * (1.0 + stream.abs().max())
