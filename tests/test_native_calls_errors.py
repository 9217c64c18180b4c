"""Errors inside the native call layer (csrc/torch_calls.cpp) come back as Python exceptions, also where the tensors' sizes or
pointers raise them: nothing may throw while the interpreter lock is released.  Fake tensors have a device and sizes and no
memory, so this runs without a GPU."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from caif_amd import torch_ops as T


@pytest.fixture
def fakes():
    with FakeTensorMode():
        f = lambda *s: torch.empty(s, device="cuda")                              # noqa: E731
        i = lambda *s: torch.empty(s, device="cuda", dtype=torch.int32)           # noqa: E731
        yield f, i


def test_expert_ids_of_one_dimension_are_refused(fakes):
    f, i = fakes
    ids, dmap, off, x, w = i(4), i(4), i(4), f(4, 16), f(4)
    for call, error in ((lambda: T.moe_dispatch(x, ids, dmap, off, 4), IndexError),
                        (lambda: T.moe_combine_backward_grad_expert(x, ids, w, dmap, off, 4), IndexError),
                        (lambda: T.moe_combine(x, ids, w, dmap, off), ValueError),
                        (lambda: T.moe_dispatch_backward(x, ids, dmap, off), ValueError),
                        (lambda: T.moe_combine_backward_grad_weights(x, x, ids, dmap, off), ValueError),
                        (lambda: T.moe_combine(f(16), i(4, 1), w, dmap, off), IndexError)):
        with pytest.raises(error):
            call()


def test_tensors_without_memory_are_an_error(fakes):
    f, i = fakes
    fw = T.FrozenWeight(f(64), T.W_F32, None, 8, 8)
    for call in (lambda: T.qlinear_forward(f(2, 8), fw, T.F32), lambda: T.qlinear_backward_input(f(2, 8), fw, T.F32),
                 lambda: T.silu(f(4)), lambda: T.multiply(f(4), f(4)), lambda: T.swiglu_backward(f(4), f(4), f(4)),
                 lambda: T.quantize_int8(f(8, 8), True), lambda: T.quantize_int8(f(8, 8), False),
                 lambda: T.quantize_int4_per_group(f(8, 128), 128), lambda: T.moe_build_dispatch_map(i(4, 2), 3),
                 lambda: T.moe_dispatch(f(4, 16), i(4, 2), i(4, 2), i(4), 8)):
        with pytest.raises(RuntimeError):
            call()
