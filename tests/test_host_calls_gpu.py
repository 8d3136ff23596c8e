"""The launches whose checks are made in C++: the same results as through the Python checks, and the same refusals."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class Absent:
    """A host module that takes nothing."""

    def __getattr__(self, name):
        return lambda *args: 0


class Counted:
    def __init__(self, real):
        self.real, self.taken = real, []

    def __getattr__(self, name):
        def call(*args):
            got = getattr(self.real, name)(*args)
            self.taken.append((name, got))
            return got
        return call


@pytest.fixture(scope="module")
def both():
    from longbow_quarrel_amd.kernels.hip import HipKernels

    fast, slow = HipKernels(), HipKernels()
    fast.host, slow.host = Counted(fast.host), Absent()
    return fast, slow


def same(both, name, call, out):
    """`call(kn, out)` on both, from equal buffers: equal results, and the host module launched for the first."""
    results = []
    for kn in both:
        o = [t.clone() for t in out]
        call(kn, o)
        results.append(o)
    assert all(torch.equal(a, b) for a, b in zip(*results))
    assert both[0].host.taken[-1] == (name, 1)


@pytest.mark.parametrize("rows,n,k,dtype,packed", [
    (1, 48, 40, torch.float32, False), (17, 2048, 2048, torch.bfloat16, True), (5, 33, 64, torch.bfloat16, False), (70, 4096, 512, torch.bfloat16, True)])
def test_products(both, rows, n, k, dtype, packed):
    gen = torch.Generator().manual_seed(n)
    x = torch.randn(rows, k + 8, generator=gen).to(dtype).cuda()[:, :k]
    w = torch.randn(n, k, generator=gen).to(dtype).cuda()
    w = both[0].pack_weight(w) if packed else w
    assert packed == bool(getattr(w, "packed", False))
    wide = torch.zeros(rows, n + 4, device="cuda")
    same(both, "linear", lambda kn, o: kn.linear(x, w, o[0][:, :n]), [wide])
    same(both, "linear", lambda kn, o: kn.linear(x, w, o[0]), [torch.zeros(rows, n, dtype=dtype, device="cuda")])
    pieces = both[0].linear_pieces(dtype, rows, n, k)
    same(both, "linear", lambda kn, o: kn.linear(x, w, o[0]), [torch.zeros(pieces, rows, n, device="cuda")])
    if dtype == torch.bfloat16 and n % 16 == 0:
        same(both, "linear_swiglu", lambda kn, o: kn.linear_swiglu(x, w, o[0]), [torch.zeros(rows, n // 2, dtype=dtype, device="cuda")])


@pytest.mark.parametrize("pieces", [None, 0, 3])
def test_norms(both, pieces):
    x, w = torch.randn(9, 96).cuda(), torch.randn(96).cuda()
    delta = None if pieces is None else torch.randn(*((pieces,) if pieces else ()), 9, 96).cuda()
    same(both, "rmsnorm", lambda kn, o: kn.rmsnorm(o[0], w, 1e-5, o[1], delta=delta), [x, torch.zeros(9, 96, dtype=torch.bfloat16, device="cuda")])


def test_a_prompt_of_attention(both):
    H, G, D, rows, BS = 4, 2, 64, 37, 64
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    pos, seq, slot, cu, table = i32(list(range(30)) + list(range(7))), i32([0] * 30 + [1] * 7), i32([1, 0]), i32([0, 30, 37]), i32([[0, 1], [2, 3]])
    freqs = (10000.0 ** (-torch.arange(D // 2, dtype=torch.float64) / (D // 2))).cuda()
    qkv = torch.randn(2, rows, (H + 2 * G) * D).cuda()
    bf = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    same(both, "rope_store_pieces", lambda kn, o: kn.rope_store_pieces(qkv, o[0], H, G, D, freqs, pos, seq, slot, table, o[1], o[2], BS),
         [bf(rows, H * D), bf(4, G, BS, D), bf(4, G, D, BS)])
    q, k, v = torch.randn(rows, H * D).bfloat16().cuda(), torch.randn(4, G, BS, D).bfloat16().cuda(), torch.randn(4, G, D, BS).bfloat16().cuda()
    same(both, "attention", lambda kn, o: kn.attention(q, o[0], H, G, D, pos, seq, slot, cu, table, k, v, BS, D ** -0.5, max_len=30), [bf(rows, H * D)])


def test_what_is_refused_stays_refused(both):
    from longbow_quarrel_amd.kernels.hip import KernelLibraryError, PackedWeight

    kn = both[0]
    x, w, out = torch.zeros(3, 64).cuda(), torch.zeros(8, 64).cuda(), torch.full((3, 8), 7.0).cuda()
    narrow = torch.zeros(4096, 64, dtype=torch.bfloat16, device="cuda")
    for args in ((x.cpu(), w, out), (x, w.bfloat16(), out), (x[:, ::2], w[:, :32], out), (x, w[:, :32], out), (x, w, out[:2]), (x, w, out.double()),
                 (x[0], w, out), (x, w, out.expand(2, 3, 8)), (x, PackedWeight(narrow, 8, 64), out)):
        with pytest.raises(KernelLibraryError):
            kn.linear(*args)
    with pytest.raises((TypeError, ValueError)):
        kn.rmsnorm(x, torch.zeros(64).cuda(), "small", torch.zeros(3, 64).cuda(), delta=torch.ones(3, 64).cuda())
    assert bool((out == 7.0).all()) and bool((x == 0.0).all())
