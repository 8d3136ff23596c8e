"""What the kernels' wrappers refuse before an address goes to a kernel: on tensors that have a device, sizes and strides but
no memory, with a library whose functions must not be called."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from longbow_quarrel_amd.kernels import hip
from longbow_quarrel_amd.kernels.hip import HipKernels, KernelLibraryError


class Untouched:
    def __getattr__(self, name):
        return lambda *args: pytest.fail(f"{name} was called")


@pytest.fixture
def kn(monkeypatch):
    monkeypatch.setattr(hip, "_ptr", lambda t: None)
    kn = object.__new__(HipKernels)
    kn.lib, kn.force_generic, kn._stream = Untouched(), False, 0
    with FakeTensorMode():
        yield kn


def on_gpu(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda:0")


def test_a_latent_layers_rows_and_their_places(kn):
    rows, q, kv, rot, block, blocks, slots = 5, 24, 16, 8, 64, 6, 2
    i32 = lambda *shape: on_gpu(*shape, dtype=torch.int32)
    bf = lambda *shape: on_gpu(*shape, dtype=torch.bfloat16)
    given = dict(src=on_gpu(rows, q + kv + rot), q_weight=on_gpu(q), cq=bf(rows, q), eps=1e-5, kv_weight=on_gpu(kv), rot_dim=rot,
                 cos_sin=on_gpu(rows, rot // 2, 2), row_pos=i32(rows), row_seq=i32(rows), seq_slot=i32(slots),
                 block_table=i32(slots, 3), kcache=bf(blocks, 1, block, kv + rot), vcache=bf(blocks, 1, kv, block), block_size=block)
    long, cpu = torch.int64, "cpu"
    for name, wrong in [
            ("seq_slot", given["seq_slot"].to(long)), ("seq_slot", given["seq_slot"].to(cpu)), ("seq_slot", i32(2 * slots)[::2]),
            ("row_pos", given["row_pos"].to(cpu)), ("row_seq", given["row_seq"].to(cpu)), ("row_pos", i32(rows - 1)),
            ("row_seq", given["row_seq"].to(long)), ("block_table", i32(slots * 3)), ("block_table", given["block_table"].to(long)),
            ("block_table", i32(slots, 6)[:, ::2]), ("vcache", bf(blocks - 1, 1, kv, block)), ("vcache", on_gpu(blocks, 1, kv, block)),
            ("kcache", bf(blocks, 1, block, kv + rot + 1)), ("kcache", bf(blocks, 1, block, kv + rot).to(cpu)),
            ("cos_sin", on_gpu(rows - 1, rot // 2, 2)), ("src", on_gpu(rows, q + kv)), ("cq", on_gpu(rows, q))]:
        with pytest.raises(KernelLibraryError):
            kn.latent_rows(**{**given, name: wrong})
    with pytest.raises(pytest.fail.Exception):  # (the whole of it comes through)
        kn.latent_rows(**given)


def test_runs_of_a_packed_weight():
    """Rows of a run of columns lie as far apart as the whole matrix's: runs of runs begin where `packed_at` says."""
    kn = object.__new__(HipKernels)
    kn.lib = hip.load_library()
    rows, cols = 4112, 1600
    whole = hip.PackedWeight(torch.arange(rows * cols).to(torch.int32).view(torch.bfloat16).view(-1)[::2].reshape(rows, cols), rows, cols)
    packed_at = lambda r, c: (r // 8 * 8) * cols + c // 64 * 512 + r % 8 * 64 + c % 64  # (8 rows' runs of 64 side by side)
    flat = whole.data.view(-1)

    def begins_at(w, r, c):
        return w.data_ptr() == flat[packed_at(r, c):].data_ptr()

    columns = kn.weight_columns(whole, 1024, 576)
    assert tuple(columns.shape) == (rows, 576) and columns.stride() == (cols, 1) and begins_at(columns, 0, 1024)
    part = kn.weight_rows(columns, 16, 2048)
    assert tuple(part.shape) == (2048, 576) and part.stride() == (cols, 1) and begins_at(part, 16, 1024)
    assert not part.is_contiguous() and kn.weight_columns(part, 0, 512) is None
    with pytest.raises(KernelLibraryError):
        part.contiguous()
    part = kn.weight_rows(whole, 2056, 2056)
    assert part.stride() == (cols, 1) and begins_at(part, 2056, 0) and part.contiguous() is part and part.data.numel() == part.numel()
    for start, n in ((4, 2048), (0, 2052), (2072, 2048), (0, 1024)):
        assert kn.weight_rows(columns, start, n) is None
