"""The names under which timed products are reported."""
import torch

from longbow_quarrel_amd.kernels.timed import TimedKernels


def test_a_product_is_named_by_its_sizes_also_over_a_run_of_weights():
    x, w = torch.zeros(6, 16), torch.zeros(4, 16)
    assert TimedKernels._label("linear", (x, w)) == "linear 6 x 4 x 16"
    assert TimedKernels._label("linear_grouped", (x, [w, w, w])) == "linear_grouped 6 x 4 x 16 of 3"
    assert TimedKernels._label("rmsnorm", (x,)) == "rmsnorm"
