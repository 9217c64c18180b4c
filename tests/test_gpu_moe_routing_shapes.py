"""The routing entry points take rows x columns and refuse other ranks."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T      # noqa: E402


def test_three_dimensional_tensors_are_refused():
    ids = torch.zeros(4, 2, dtype=torch.int32, device="cuda")
    dmap, off = T.moe_build_dispatch_map(ids, 3)
    x, w = torch.zeros(4, 1, 16, device="cuda"), torch.zeros(4, 2, device="cuda")
    ids3 = ids.reshape(4, 2, 1)
    buf = torch.zeros(8, 16, device="cuda")
    for call in (lambda: T.moe_dispatch(x, ids, dmap, off, 8), lambda: T.moe_combine(buf, ids3, w, dmap, off),
                 lambda: T.moe_combine_backward_grad_expert(x, ids, w, dmap, off, 8), lambda: T.moe_dispatch_backward(buf, ids3, dmap, off),
                 lambda: T.moe_combine_backward_grad_weights(buf[:4], buf, ids3, dmap, off)):
        with pytest.raises(ValueError):
            call()
