"""Expert buffers that hold nothing yet (caifx_moe_dispatch_fresh, caifx_moe_combine_backward_grad_expert_fresh): the same bytes as clearing
the buffer and filling it, nothing around it touched."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T      # noqa: E402


# rows that are not a multiple of a 16-byte piece; one row and the most that the filling launch looks after (1024, of as many assignments
# at most), and beyond; dropped and invalid assignments, rows in front of the first segment and behind the last
@pytest.mark.parametrize("tokens,top_k,experts,dim,extra,capacity,dtype", [
    (1, 1, 3, 1, 0, 0, torch.float32), (1, 2, 3, 7, 40, 0, torch.bfloat16), (16, 6, 64, 2048, 0, 0, torch.bfloat16),
    (37, 3, 8, 24, 5, 4, torch.float16), (251, 4, 16, 33, 20, 50, torch.float32), (256, 4, 64, 256, 0, 9, torch.bfloat16),
    (513, 2, 8, 8, 3, 0, torch.bfloat16), (64, 2, 4, 1, 897, 0, torch.float32), (3000, 6, 64, 256, 5, 200, torch.bfloat16)])
def test_rows_without_an_assignment_are_zero(tokens, top_k, experts, dim, extra, capacity, dtype):
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    ids = torch.randint(-1, experts + 1, (tokens, top_k), device="cuda", dtype=torch.int32, generator=gen)
    dmap, offsets = T.moe_build_dispatch_map(ids, experts, capacity)
    if extra >= 3:
        offsets = offsets + 3                                                    # rows in front of the first segment
    rows = tokens * top_k + extra
    x = torch.empty(tokens, dim, device="cuda").normal_(generator=gen).to(dtype)
    w = torch.rand(tokens, top_k, device="cuda", generator=gen).to(dtype)
    pad = 5
    for grad in (False, True):
        def fill(buf, entry, *more):
            head = (x.data_ptr(), ids.data_ptr()) + ((w.data_ptr(),) if grad else ())
            capi.call(entry, *head, dmap.data_ptr(), offsets.data_ptr(), buf.data_ptr(), *more, tokens, dim, top_k, experts, T.CODE_OF[dtype], None)
        entry = "caifx_moe_combine_backward_grad_expert" if grad else "caifx_moe_dispatch"
        want = torch.zeros(rows, dim, device="cuda", dtype=dtype)
        fill(want, entry)
        got = torch.full((pad + rows * dim + pad,), float("nan"), device="cuda", dtype=dtype)
        torch.cuda.synchronize()
        fill(got[pad:], entry + "_fresh", rows)
        torch.cuda.synchronize()
        assert torch.equal(got[pad:pad + rows * dim].reshape(rows, dim), want)
        assert bool(got[:pad].isnan().all()) and bool(got[pad + rows * dim:].isnan().all())
        op = (lambda *a: T.moe_combine_backward_grad_expert(x, ids, w, *a)) if grad else (lambda *a: T.moe_dispatch(x, ids, *a))
        assert torch.equal(op(dmap, offsets, rows), want)


def test_no_tokens():
    ids = torch.empty((0, 2), dtype=torch.int32, device="cuda")
    dmap, offsets = T.moe_build_dispatch_map(ids, 4)
    x = torch.empty((0, 24), device="cuda")
    assert not T.moe_dispatch(x, ids, dmap, offsets, 9).any()
    assert T.moe_dispatch(x, ids, dmap, offsets, 0).shape == (0, 24)
