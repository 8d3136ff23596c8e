"""Gated linear attention in chunks of 64 tokens, against the recurrence in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TAU = 16.0


def case(H, dk, dv, lengths, seed, pad=0):
    """q, k, v, z [rows, .] (with `pad` columns behind each), bias, starting states [slots, H, dv, dk]."""
    g = torch.Generator().manual_seed(seed)
    rows = sum(lengths)
    wide = lambda n, m, s: torch.empty(rows, n + pad).normal_(m, s, generator=g)
    return (wide(H * dk, 0, 1), wide(H * dk, 0, 1), wide(H * dv, 0, 1), wide(H * dk, 1, 2),
            torch.empty(H * dk).normal_(2, 2, generator=g), torch.empty(len(lengths) + 1, H, dv, dk).normal_(0, 1, generator=g))


def plain(x, H, dk, dv, lengths):
    q, k, v, z, bias, start = (t.double() for t in x)
    out, ends, at = torch.empty(sum(lengths), H * dv, dtype=torch.float64), [], 0
    a = torch.sigmoid(z[:, : H * dk] + bias).pow(1 / TAU).view(-1, H, dk)
    for b, n in enumerate(lengths):
        S = start[b + 1].transpose(1, 2).clone()
        for r in range(at, at + n):
            S = a[r][:, :, None] * S + k[r, : H * dk].view(H, dk)[:, :, None] * v[r, : H * dv].view(H, dv)[:, None, :]
            out[r] = (S * (q[r, : H * dk].view(H, dk) * dk ** -0.5)[:, :, None]).sum(1).reshape(-1)
        ends.append(S.transpose(1, 2))
        at += n
    return out, torch.stack(ends)


def run(x, H, dk, dv, lengths, chunked, scratch=None):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    q, k, v, z, bias, start = (t.cuda() for t in x)
    rows, batch = sum(lengths), len(lengths)
    cu = torch.tensor([sum(lengths[:b]) for b in range(batch + 1)], dtype=torch.int32, device="cuda")
    slots = torch.arange(1, batch + 1, dtype=torch.int32, device="cuda")
    out, state, more = torch.full((rows, H * dv), 7.0, device="cuda"), start.clone(), {}
    if chunked:
        need = kn.gla_chunks_workspace(rows, batch, H, dk, dv, max(lengths))
        assert need > 0
        more = dict(max_rows=max(lengths), chunked=True, workspace=torch.full((scratch or need,), float("nan"), device="cuda"))
    kn.gla_scan(q[:, : H * dk], k[:, : H * dk], v[:, : H * dv], z[:, : H * dk], bias, state, out, H, dk, dv, dk ** -0.5, 1 / TAU,
                slots, cu, batch, **more)
    assert torch.equal(state[0].cpu(), x[5][0])
    return out.cpu(), state[1:].cpu()


def err(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("H,dk,dv,lengths,pad", [
    (2, 128, 256, [2048], 0), (1, 128, 33, [64], 0), (3, 17, 9, [65, 1, 300], 0), (2, 64, 24, [63, 64, 128, 129], 3),
    (1, 100, 33, [1] * 70 + [191], 4), (8, 128, 40, [300, 310], 0)])
def test_chunks(H, dk, dv, lengths, pad):
    x = case(H, dk, dv, lengths, sum(lengths) + dk, pad)
    want, ends = plain(x, H, dk, dv, lengths)
    walked, walked_end = run(x, H, dk, dv, lengths, False)
    got, end = run(x, H, dk, dv, lengths, True)
    # no further from 64 bits than the walk token by token, or than the 64 roundings of 2^-24 of a chunk's products of decays
    assert err(got, want) < max(err(walked, want), 64 * 2.0 ** -24) and err(end, ends) < max(err(walked_end, ends), 64 * 2.0 ** -24)
    print("errors: chunks", err(got, want), err(end, ends), "walk", err(walked, want), err(walked_end, ends))


def test_rounds_of_chunks_leave_the_same_bits():
    H, dk, dv, lengths = 2, 32, 48, [200, 70, 500]
    x = case(H, dk, dv, lengths, 5)
    from longbow_quarrel_amd.kernels.hip import HipKernels

    one = HipKernels().lib.lq_delta_scan_least
    import ctypes

    one.restype = ctypes.c_longlong
    whole, end = run(x, H, dk, dv, lengths, True)
    parts, parts_end = run(x, H, dk, dv, lengths, True, scratch=2 * int(one(ctypes.c_int(H))))
    assert torch.equal(whole, parts) and torch.equal(end, parts_end)


@pytest.mark.parametrize("where", ["q", "k", "v", "z"])
def test_a_nan_reaches_no_earlier_token(where):
    H, dk, dv, lengths, at = 1, 32, 32, [150], 77
    x = list(case(H, dk, dv, lengths, 9))
    clean, _ = run(x, H, dk, dv, lengths, True)
    x["qkvz".index(where)] = x["qkvz".index(where)].clone()
    x["qkvz".index(where)][at] = float("nan")
    got, _ = run(x, H, dk, dv, lengths, True)
    assert torch.equal(got[:at], clean[:at]) and got[at].isnan().all()
