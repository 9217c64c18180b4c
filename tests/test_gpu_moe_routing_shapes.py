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


def test_more_tokens_than_eight_waves_each_fit_a_grid():
    # 8.4 million tokens of 449 values: eight waves a token would be 2^32 threads
    tokens, dim, rows = 8_500_000, 449, 16
    buf = torch.randn(rows, dim, device="cuda").to(torch.bfloat16)
    ids = torch.zeros(tokens, 1, dtype=torch.int32, device="cuda")
    dmap = (torch.arange(tokens, device="cuda", dtype=torch.int32) % rows).reshape(tokens, 1)
    off = torch.tensor([0, rows], dtype=torch.int32, device="cuda")
    ones = torch.ones(tokens, 1, device="cuda", dtype=torch.bfloat16)
    for call in (lambda: T.moe_combine(buf, ids, ones, dmap, off), lambda: T.moe_dispatch_backward(buf, ids, dmap, off)):
        y = call()
        last = buf[dmap[-1000:, 0].long()]
        assert torch.equal(y[-1000:], last) and torch.equal(y[:rows], buf)
        assert torch.equal(y[:tokens // rows * rows].reshape(-1, rows, dim).amax(0), buf)
        del y
