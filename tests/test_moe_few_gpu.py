"""A mixture of experts over few rows, reading the chosen experts' weights alone, against the formula in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def weighted(gate, up, w, activation, on_input, limit):
    """An expert's activations [rows, ff] in float64 (gate is None for the square of relu)."""
    if activation == "relu2":
        return torch.relu(up) ** 2 * w
    s = w if on_input else torch.ones_like(w)
    gate, up = gate * s, up * s
    if activation == "silu":
        y = gate * torch.sigmoid(gate) * up
    else:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
        y = gate * torch.sigmoid(1.702 * gate) * (up + 1)
    return y if on_input else y * w


@pytest.mark.parametrize("rows,E,top,ff,shared,width,activation,more", [
    (1, 8, 2, 64, 0, 512, "clamped_swish", dict(on_input=True, limit=1.0)),
    (8, 8, 2, 3584, 0, 2048, "clamped_swish", dict(on_input=True, limit=7.0)),
    (16, 4, 1, 192, 128, 576, "silu", dict(gate=True)),
    (7, 6, 2, 2560, 2048, 2048, "silu", dict(gate=True, passed=2)),
    (3, 64, 3, 64, 64, 4096, "silu", dict(on_input=True)),
    (16, 64, 4, 128, 0, 1536, "relu2", {}),
    (9, 8, 8, 320, 1344, 2112, "relu2", dict(passed=1)),
    (2, 5, 0, 64, 0, 512, "silu", {}),            # nobody chose anything
    (5, 5, 0, 128, 64, 640, "silu", dict(passed=3)),
    (8, 3, 1, 512, 640, 2048, "silu", {}), (6, 3, 2, 576, 512, 2560, "relu2", {}), (13, 3, 2, 640, 0, 3072, "silu", {}),
    (1, 1, 1, 64, 0, 512, "relu2", {})])
@pytest.mark.parametrize("pack", [True, False])
def test_chosen_experts_alone(rows, E, top, ff, shared, width, activation, more, pack):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    kn.pack_weights = pack
    gen = torch.Generator().manual_seed(rows * 1000 + ff + E)
    parts = 1 if activation == "relu2" else 2
    inner = E * ff + shared
    x = torch.randn(rows, width, generator=gen).bfloat16()
    w_in = (torch.randn(inner * parts, width, generator=gen) * width ** -0.5).bfloat16()
    w_out = (torch.randn(width, inner, generator=gen) * 0.02).bfloat16()
    route = torch.full((rows, E), -1.0)
    for r in range(rows):
        route[r, torch.randperm(E, generator=gen)[:top]] = torch.rand(top, generator=gen) + 0.1
    gate = torch.randn(rows, 4, generator=gen)[:, 1:2] if more.get("gate") else None
    passed = torch.rand(rows, more["passed"], generator=gen) - 0.5 if "passed" in more else None
    if passed is not None:
        passed[passed < 0] = -1.0
    nobody = [e for e in range(E) if (route[:, e] < 0).all()]
    poisoned_in, poisoned_out = w_in.clone(), w_out.clone()  # what nobody chose is not read
    for e in nobody:
        poisoned_in[e * parts * ff : (e + 1) * parts * ff] = float("nan")
        poisoned_out[:, e * ff : (e + 1) * ff] = float("nan")
    assert kn.moe_few_supported(torch.bfloat16, rows, E, ff, shared, width)

    act64 = torch.zeros(rows, inner, dtype=torch.float64)
    for e in range(E + (1 if shared else 0)):
        n, at = (ff, e * ff) if e < E else (shared, E * ff)
        y = x.double() @ w_in[at * parts : (at + n) * parts].double().T
        if e < E:
            w = route[:, e : e + 1].double()
            v = weighted(y[:, :n] if parts == 2 else None, y[:, (parts - 1) * n :], w, activation, more.get("on_input", False),
                         more.get("limit", 0.0))
            act64[:, at : at + n] = torch.where(w >= 0, v, 0.0)
        else:
            one = torch.ones(rows, 1, dtype=torch.float64)
            v = weighted(y[:, :n] if parts == 2 else None, y[:, (parts - 1) * n :], one, activation, False, 0.0)
            act64[:, at : at + n] = v * (torch.sigmoid(gate.double()) if gate is not None else 1.0)
    want = act64 @ w_out.double().T
    bound = 2.0 ** -8 * (act64.abs() @ w_out.double().abs().T)  # (an activation's rounding to 8 bits: half of this; sums: 2^-24 a term)
    if passed is not None:
        share = passed.clamp(min=0).double().sum(1, keepdim=True) * x.double()
        want, bound = want + share, bound + 2.0 ** -22 * share.abs()

    held, second = kn.pack_weight(poisoned_in.cuda()), kn.pack_weight(poisoned_out.cuda())
    act = torch.full((rows, inner), 7.0, dtype=torch.bfloat16, device="cuda")
    pieces = kn.moe_few_pieces(width) if rows % 2 else (1, 2, 4)[rows // 2 % 3]
    out = torch.full((pieces, rows, width), 7.0, device="cuda")
    kn.moe_few(x.cuda(), held, second, route.cuda(), act, out, ff, shared, activation, limit=more.get("limit", 0.0),
               on_input=more.get("on_input", False), shared_gate=gate.cuda() if gate is not None else None,
               passed=passed.cuda() if passed is not None else None)
    assert ((out.double().sum(0).cpu() - want).abs() <= bound + 1e-30).all()
    for e in nobody:
        assert (act[:, e * ff : (e + 1) * ff] == 7.0).all()
    if rows > 1 and top:  # a row's bits do not depend on what the others chose
        alone = torch.full((rows, E), -1.0)
        alone[0] = route[0]
        again = torch.empty_like(out)
        kn.moe_few(x.cuda(), held, second, alone.cuda(), act, again, ff, shared, activation, limit=more.get("limit", 0.0),
                   on_input=more.get("on_input", False), shared_gate=gate.cuda() if gate is not None else None,
                   passed=passed.cuda() if passed is not None else None)
        assert torch.equal(again[:, 0], out[:, 0])


@pytest.mark.parametrize("ff,shared,width", [(64, 0, 512), (64, 64, 1088), (2112, 0, 1024), (4160, 64, 576), (10304, 0, 2112)])
@pytest.mark.parametrize("activation", ["silu", "relu2"])
@pytest.mark.parametrize("apart", [0, 72])
def test_first_product_of_any_number_of_tiles(ff, shared, width, activation, apart):
    """Workgroups of none, one, an odd and an even number of tiles, wavefronts without a share of K, and a dense weight's rows apart."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, rows, E = HipKernels(), 3, 2
    gen = torch.Generator().manual_seed(ff + width)
    parts, inner = 1 if activation == "relu2" else 2, E * ff + shared
    x = torch.randn(rows, width, generator=gen).bfloat16()
    wide = torch.full((inner * parts, width + apart), float("nan"), dtype=torch.bfloat16)
    w_in = wide[:, :width]
    w_in.copy_(torch.randn(inner * parts, width, generator=gen) * width ** -0.5)
    route = torch.tensor([[0.5, -1.0], [0.25, 0.75], [-1.0, 1.0]])
    act = torch.full((rows, inner), 7.0, dtype=torch.bfloat16, device="cuda")
    w_out = torch.zeros(width, inner, dtype=torch.bfloat16, device="cuda")
    out = torch.empty(1, rows, width, device="cuda")
    kn.pack_weights = apart == 0
    held = wide.cuda()[:, :width] if apart else kn.pack_weight(w_in.contiguous().cuda())
    kn.moe_few(x.cuda(), held, w_out, route.cuda(), act, out, ff, shared, activation)
    for e in range(E + (1 if shared else 0)):
        n, at = (ff, e * ff) if e < E else (shared, E * ff)
        y = x.double() @ w_in[at * parts : (at + n) * parts].double().T
        w = route[:, e : e + 1].double() if e < E else torch.ones(rows, 1, dtype=torch.float64)
        v = weighted(y[:, :n] if parts == 2 else None, y[:, (parts - 1) * n :], w, activation, False, 0.0)
        want = torch.where(w >= 0, v, 0.0)
        # (half a unit of 8 bits at the result; the sums' 2^-24 a term of at most 2 112 at the products' size, times the factors beside them)
        bound = 2.0 ** -8 * want.abs() + 2112 * 2.0 ** -24 * 16.0
        assert ((act[:, at : at + n].double().cpu() - want).abs() <= bound).all()


@pytest.mark.parametrize("rows,ff,places", [
    (8, 2176, (0, 64, 2048)),     # a wavefront's chunks 0 and 16 of 128 k: the sums of their halves are apart
    (1, 2176, (100, 40, 2148)),
    (9, 2048, (0, 64, 1024)),     # chunks of 64 k: 0 and 16 are one wavefront's, 1 another's
    (8, 1088, (3, 67, 1027))])
@pytest.mark.parametrize("pack", [True, False])
def test_sums_of_halves_and_chunks_stay_apart(rows, ff, places, pack):
    """2^24 + 1 - 2^24 at three places of the second product's k: one where the two large ones are of one sum and the one of another,
    nothing where a sum takes the one between them."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, width = HipKernels(), 4096
    kn.pack_weights = pack
    assert kn.moe_few_pieces(width) == 1 and kn.moe_few_supported(torch.bfloat16, rows, 1, ff, 0, width)
    w_in = torch.zeros(ff, width, dtype=torch.bfloat16)
    w_out = torch.zeros(width, ff, dtype=torch.bfloat16)
    for k, v in zip(places, (2.0 ** 24, 1.0, -2.0 ** 24)):
        w_in[k, 0], w_out[:, k] = 1.0, v  # (relu(1)^2 is 1)
    x = torch.ones(rows, width, dtype=torch.bfloat16)
    act, out = torch.empty(rows, ff, dtype=torch.bfloat16, device="cuda"), torch.empty(rows, width, device="cuda")
    kn.moe_few(x.cuda(), kn.pack_weight(w_in.cuda()), kn.pack_weight(w_out.cuda()), torch.ones(rows, 1, device="cuda"), act, out,
               ff, 0, "relu2")
    assert bool((out == 1.0).all())


@pytest.mark.parametrize("rows,ff,width", [(8, 128, 512), (8, 576, 2048), (12, 704, 2112)])
@pytest.mark.parametrize("pack", [True, False])
def test_activations_beyond_32_bit_offsets(rows, ff, width, pack):
    """Rows of activations 2^31 bytes from first to last and more: the bits of the same ones side by side."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, E, shared = HipKernels(), 3, 64
    kn.pack_weights = pack
    gen = torch.Generator(device="cuda").manual_seed(rows + ff)
    inner, apart = E * ff + shared, 2 ** 31 // 2 // (rows - 1) // 8 * 8 + 8
    x, w_in = (torch.randn(n, width, generator=gen, device="cuda").bfloat16() for n in (rows, inner))
    w_out = torch.randn(width, inner, generator=gen, device="cuda").bfloat16()
    route = torch.rand(rows, E, generator=gen, device="cuda")
    route[:, 1], route[0, 2] = -1.0, -1.0
    outs = []
    for act in (torch.empty(rows, inner, dtype=torch.bfloat16, device="cuda"),
                torch.empty((rows - 1) * apart + inner, dtype=torch.bfloat16, device="cuda").as_strided((rows, inner), (apart, 1))):
        out = torch.empty(kn.moe_few_pieces(width), rows, width, device="cuda")
        kn.moe_few(x, kn.pack_weight(w_in), kn.pack_weight(w_out), route, act, out, ff, shared, "relu2")
        outs.append(out)
    assert torch.equal(*outs)


def test_how_many_columns_are_taken():
    """Up to 2^30 columns of the second matrix, as offsets of its rows are 64-bit where they have to be."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    assert kn.moe_few_supported(torch.bfloat16, 8, 64, 2 ** 20, 0, 512) and kn.moe_few_supported(torch.bfloat16, 16, 16, 2 ** 26 - 64, 64, 4096)
    assert not kn.moe_few_supported(torch.bfloat16, 8, 64, 2 ** 24, 0, 512)


def test_sizes_that_are_not_taken():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    take = lambda *a: kn.moe_few_supported(torch.bfloat16, *a)
    assert take(16, 64, 64, 0, 512) and not take(17, 8, 64, 0, 512) and not take(1, 65, 64, 0, 512)
    assert not take(1, 8, 96, 0, 512) and not take(1, 8, 64, 32, 512) and not take(1, 8, 64, 0, 448) and not take(1, 8, 64, 0, 4160)
    assert not kn.moe_few_supported(torch.float32, 1, 8, 64, 0, 512)
