"""Products of at most 16 rows whose weights go through LDS: runs of one, several and half tiles of columns, shares of K of no, one and
several slabs of 64, in full runs and what is left, every way out; dense and packed weights the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(8, 2560), (2048, 512), (2048, 4160), (2056, 960), (2064, 1024), (3080, 1088), (4096, 64 * 16 * 5), (6160, 4096), (10248, 576),
         (28688, 1216), (40960, 512), (2048, 14400), (4104, 12352), (32784, 2048)]


def halves(values, bounds):
    """Gate's and up's columns, interleaved in eights, each with its bound."""
    parts = [t.reshape(len(t), -1, 2, 8).unbind(2) for t in (values, bounds)]
    return [tuple(p[i].reshape(len(values), -1) for p in parts) for i in (0, 1)]


@pytest.mark.parametrize("rows", [1, 3, 8, 12, 16])
@pytest.mark.parametrize("n,k", SIZES)
def test_every_way_out(rows, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x = torch.randn(rows, k + 8, generator=gen, device="cuda").to(bf)[:, :k]
    w = torch.randn(n, k, generator=gen, device="cuda").to(bf)
    want, terms = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bound = k * 2.0 ** -24 * terms  # (products of bfloat16 are exact in 32 bits; a rounding a term, in any order)
    got = []
    for held in (w, kn.pack_weight(w)):
        wide = torch.full((rows + 1, n + 5), 7.0, device="cuda")
        kn.linear(x, held, wide[:rows, :n])
        assert ((wide[:rows, :n] - want).abs() <= bound).all() and bool((wide[rows] == 7).all()) and bool((wide[:, n:] == 7).all())
        narrow = torch.empty(rows, n, dtype=bf, device="cuda")
        kn.linear(x, held, narrow)
        assert ((narrow - want).abs() <= bound + 2.0 ** -8 * want.abs()).all()
        outs = [wide, narrow]
        if n % 16 == 0 and n >= 2048:
            gated = torch.empty(rows, n // 2, dtype=bf, device="cuda")
            kn.linear_swiglu(x, held, gated, activation="relu")
            gate, up = wide[:rows, :n].reshape(rows, n // 16, 2, 8).unbind(2)
            (g, off_g), (u, off_u) = halves(want, bound)
            assert ((gated - g.clamp(min=0) * u).abs() <= 1.001 * (off_g * (u.abs() + off_u) + g.abs() * off_u) + 2.0 ** -8 * (g * u).abs()).all()
            # (2 048 columns and 13 rows and more: the whole product may take another kernel, whose sums have another order)
            assert rows > 12 or n <= 2048 or torch.equal(gated, (gate.clamp(min=0) * up).reshape(rows, n // 2).to(bf))
            outs.append(gated)
        parts = kn.linear_fused_parts(bf, rows, n, k)
        if parts:
            stream = torch.randn(rows, n, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
            gain = torch.linspace(-1, 1, n, device="cuda")
            sq, scaled, new = torch.empty(rows, parts, device="cuda"), torch.empty(rows, n, dtype=bf, device="cuda"), stream.clone()
            kn.linear_residual(x, held, new, sq, gain=gain, scaled=scaled)
            assert ((new - stream - want).abs() <= bound + 2.0 ** -23 * (stream.abs() + want.abs())).all()
            assert torch.equal(scaled, (new * gain).to(bf))
            assert ((sq.double().sum(1) - (new.double() ** 2).sum(1)).abs() <= n * 2.0 ** -24 * (new.double() ** 2).sum(1)).all()
            sums = torch.rand(rows, 300, generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
            half = torch.empty(rows, n, dtype=bf, device="cuda")
            kn.linear_scaled(x, sums, 1e-5, held, half)
            rstd = (sums.double().sum(1, keepdim=True) / k + 1e-5).rsqrt()
            assert ((half - want * rstd).abs() <= rstd * (bound + 2.0 ** -8 * want.abs()) * 1.001).all()
            outs += [new, sq, scaled, half]
            if n % 16 == 0:
                both = torch.empty(rows, n // 2, dtype=bf, device="cuda")
                kn.linear_scaled(x, sums, 1e-5, held, both, swiglu=True)
                (g, off_g), (u, off_u) = halves(want * rstd, (bound + 2.0 ** -22 * want.abs()) * rstd)  # (the root, and the product with it)
                silu = g * torch.sigmoid(g)
                # (silu' is below 1.1; the exponential and the reciprocal are off by an ulp or so, the exponent by 2^-23 of |gate|)
                off = 1.1 * off_g * (u.abs() + off_u) + silu.abs() * off_u + (4 + g.abs()) * 2.0 ** -23 * (silu * u).abs()
                assert ((both - silu * u).abs() <= 1.01 * off + 2.0 ** -8 * (silu * u).abs() + 1e-30).all()
                outs.append(both)
        got.append(outs)
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("rows,n,k", [(8, 4096, 4096), (5, 2056, 2048), (1, 28672, 1024)])
def test_an_infinity_or_nan_stays_in_its_row_or_column(rows, n, k):
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn = HipKernels()
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x, w = (torch.randn(r, k, generator=gen, device="cuda").bfloat16() for r in (rows, n))
    want, out = torch.empty(rows, n, device="cuda"), torch.empty(rows, n, device="cuda")
    kn.linear(x, w, want)
    x[0, k - 1], w[n - 1, 3] = float("inf"), float("nan")
    for held in (w, kn.pack_weight(w)):
        kn.linear(x, held, out)
        assert not bool(out[0].isfinite().any()) and bool(out[:, n - 1].isnan().all())
        assert torch.equal(out[1:, : n - 1], want[1:, : n - 1])


@pytest.mark.parametrize("rows,n,k", [(12, 4096, 1024), (3, 2048, 4096), (16, 2048, 576)])
def test_rows_of_x_beyond_32_bit_offsets(rows, n, k):
    """Rows 2^28 bytes apart and more: the bits of the same rows side by side, dense and packed, every way out."""
    from longbow_quarrel_amd.kernels.hip import HipKernels

    kn, bf = HipKernels(), torch.bfloat16
    apart = 2 ** 31 // 2 // (rows - 1) // 8 * 8
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    near, w = (torch.randn(r, k, generator=gen, device="cuda").to(bf) for r in (rows, n))
    far = torch.empty((rows - 1) * apart + k, dtype=bf, device="cuda").as_strided((rows, k), (apart, 1))
    far.copy_(near)
    assert ((rows - 1) * apart + k) * 2 >= 2 ** 31
    stream = torch.randn(rows, n, generator=gen, device="cuda")
    gain, sums = torch.linspace(-1, 1, n, device="cuda"), torch.rand(rows, 300, generator=gen, device="cuda")
    parts = kn.linear_fused_parts(bf, rows, n, k)
    for held in (w, kn.pack_weight(w)):
        got = []
        for x in (near, far):
            wide, gated, acted, half = (torch.empty(rows, c, dtype=d, device="cuda") for c, d in
                                        ((n, torch.float32), (n // 2, bf), (n, bf), (n, bf)))
            kn.linear(x, held, wide)
            kn.linear_swiglu(x, held, gated)
            kn.linear_unit(x, held, acted, "relu2")
            biased = torch.empty(rows, n // 2 + 8, dtype=bf, device="cuda")
            kn.linear_unit(x, held, biased, "silu", bias=gain, tail=8)
            got.append([wide, gated, acted, biased])
            if parts:
                new, sq, scaled = stream.clone(), torch.empty(rows, parts, device="cuda"), torch.empty(rows, n, dtype=bf, device="cuda")
                kn.linear_residual(x, held, new, sq, gain=gain, scaled=scaled)
                kn.linear_scaled(x, sums, 1e-5, held, half)
                got[-1] += [new, sq, scaled, half]
        assert all(torch.equal(a, b) for a, b in zip(*got))
