"""The router's kernels around the numbers of experts where a lane takes one more output (64, 256, 1024), against the
choice made one expert after the other."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kn():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    return HipKernels()


def best_of(values):
    """Index of the largest of {index: value}; the first stays where the others are equal or no number is larger."""
    best = None
    for i, v in values.items():
        if best is None or v > values[best]:
            best = i
    return best


def plain(z, top, renorm, corr, groups, keep, softmax, by_max):
    """One row in float64 -> weights, -1 where not chosen."""
    E = len(z)
    if softmax:
        big = max((v for v in z if v == v), default=-math.inf)
        ex = [math.exp(v - big) if v == v else math.nan for v in z]
        s = [v / sum(ex) for v in ex]
    else:
        s = [1.0 / (1.0 + math.exp(-v)) if v == v else math.nan for v in z]
    c = [a + b for a, b in zip(s, corr)] if corr is not None else s
    allowed = range(E)
    if groups > 1 and keep < groups:
        per, marks = E // groups, {}
        for g in range(groups):
            two = sorted((v for v in c[g * per:(g + 1) * per] if v == v), reverse=True)[:2] + [-math.inf] * 2
            marks[g] = two[0] + two[1] if per > 1 and not by_max else two[0]
        kept = set()
        for _ in range(keep):
            g = best_of(marks)
            kept.add(g)
            del marks[g]
        allowed = [e for e in allowed if e // per in kept]
    left, out = {e: c[e] for e in allowed}, [-1.0] * E
    total = 0.0
    for _ in range(min(top, len(left))):
        e = best_of(left)
        del left[e]
        out[e] = s[e] if s[e] == s[e] else 0.0
        total += out[e]
    if renorm and total > 0:
        out = [v / total if v >= 0 else v for v in out]
    return out


@pytest.mark.parametrize("E,top,groups,keep,ident", [
    (1, 1, 0, 0, 0), (2, 2, 2, 1, 0), (63, 8, 0, 0, 0), (64, 8, 8, 3, 0), (64, 3, 64, 5, 0), (65, 4, 5, 2, 7), (128, 8, 64, 9, 0),
    (256, 8, 8, 4, 0), (257, 5, 0, 0, 1), (1024, 16, 64, 7, 24), (1025, 3, 5, 2, 0)])
@pytest.mark.parametrize("softmax", [False, True])
def test_choice_and_weights(kn, E, top, groups, keep, ident, softmax):
    rows = 5  # one more than a workgroup of four wavefronts has
    g = torch.Generator().manual_seed(E + top)
    # Logits and corrections in steps of 1/4 and 1/8: many exact ties, which the lower index wins, and otherwise scores too
    # far apart for 32-bit rounding to turn the order, for the tests of one score; one row has an entry that is no number
    z = (torch.randint(-12, 13, (rows, E), generator=g) / 4.0).float()
    if not softmax:
        z[1, E // 2] = math.nan
        z[2, 0] = math.nan
    for by_max, renorm in ((True, False), (False, True)):
        # (sums of two scores can be closer than their rounding: these groups are marked by scores of one power of two)
        zz = z if by_max else torch.where(z == z, torch.zeros_like(z), z)
        corr = None if by_max else torch.randint(-7, 8, (E,), generator=g) / 8.0
        if softmax and not by_max:
            zz[:, E // 2:] = -200.0  # scores of 0, and of 1 / the number of the others
        route = torch.full((rows, E - ident), -7.0, device="cuda")
        idt = torch.full((rows, ident), -7.0, device="cuda") if ident else None
        kn.moe_route(zz.cuda(), route, top, renorm, correction=corr.float().cuda() if corr is not None else None, groups=groups,
                     keep=keep, scoring="softmax" if softmax else "sigmoid", group_mark="max" if by_max else "top2",
                     identity=idt)
        got = torch.cat([route, idt], 1).cpu() if ident else route.cpu()
        for r in range(rows):
            want = plain(zz[r].double().tolist(), top, renorm, corr.tolist() if corr is not None else None, groups, keep, softmax,
                         by_max)
            w = torch.tensor(want, dtype=torch.float64)
            assert torch.equal(got[r] >= 0, w >= 0), (r, by_max)
            # a score: exp, an addition or a sum of E terms, a division; then a sum of `top` and a division more
            assert torch.allclose(got[r].double(), w, rtol=(E + top + 8) * 2.0 ** -24, atol=1e-30), (r, by_max)


@pytest.mark.parametrize("rows,K,E,extra", [(1, 8, 1, 0), (3, 520, 8, 1), (8, 2048, 8, 0), (16, 4096, 17, 0), (5, 1000, 63, 1), (2, 256, 64, 0)])
@pytest.mark.parametrize("scoring", ["sigmoid", "softmax", "softmax_chosen"])
def test_the_product_and_the_choice_in_one_launch(kn, rows, K, E, extra, scoring):
    """Its logits against 64 bits, and the choice that `moe_route` makes of them, bit for bit; rows apart by more than K."""
    gen = torch.Generator(device="cuda").manual_seed(rows + K + E)
    h, w = (torch.randn(n, K + 8, generator=gen, device="cuda").bfloat16()[:, :K] for n in (rows, E + extra))
    assert kn.moe_router_takes(torch.bfloat16, rows, K, E + extra) and not kn.moe_router_takes(torch.float32, rows, K, E)
    options = dict(scoring=scoring)
    if scoring != "softmax_chosen" and E % 8 == 0:
        options.update(correction=torch.randn(E, generator=gen, device="cuda"), groups=4, keep=2, renormalize_eps=1e-20,
                       identity=torch.full((rows, 2), 7.0, device="cuda"))
    R, top = E - (2 if "identity" in options else 0), min(E, 2)
    z = torch.full((rows, E + extra + 3), 7.0, device="cuda")
    route, want = (torch.full((rows, R), 7.0, device="cuda") for _ in range(2))
    kn.moe_router(h, w, z[:, : E + extra], E, route, top, True, **options)
    assert bool((z[:, E + extra :] == 7).all())
    # K exact products of bfloat16, in any order: at most K roundings of 2^-24 of their absolute sum
    exact, terms = h.double() @ w.double().T, h.double().abs() @ w.double().abs().T
    assert bool(((z[:, : E + extra] - exact).abs() <= K * 2.0 ** -24 * terms).all())
    passed = options.pop("identity", None)
    if passed is not None:
        options["identity"] = torch.empty_like(passed)
    kn.moe_route(z[:, :E], want, top, True, **options)
    assert torch.equal(route, want) and (passed is None or torch.equal(passed, options["identity"]))


def test_large_routers_go_in_two_launches(kn):
    """One launch reads the whole weight a row by one compute unit: it is taken for as much as that pays for."""
    pays = lambda rows, K, N: kn.moe_router_pays(torch.bfloat16, rows, K, N)
    assert pays(1, 2048, 8) and pays(8, 3072, 16) and pays(16, 7168, 16) and pays(9, 2048, 32)
    assert not (pays(8, 2048, 64) or pays(1, 4096, 32) or pays(1, 7168, 8) or pays(16, 4096, 32) or pays(17, 2048, 8) or pays(16, 256, 64))
