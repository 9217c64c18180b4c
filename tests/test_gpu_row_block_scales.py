"""int8 row-block decode kernel: every wave stages the scales of its own k range, and fp32 activations of one group per wave
stay in registers.  Against the quantised weight in 64 bits, where waves are left without a group, scale vectors are shorter
than a wave's stride or wrap inside it, and rows hold no numbers."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T      # noqa: E402

# The activations' three digits carry 2^-21 of the largest |x * scale| of a wave's k range (about four standard deviations of a
# uniform share of the terms), so the sums are off by some 2^-21 * 4 / sqrt(3) of their own size: 1.1e-6; four times that.
BOUND = 4.5e-6


def _weight(N, K, period, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    codes = torch.randint(-128, 128, (N * K,), device="cuda", generator=g, dtype=torch.int8)
    scales = None
    if period:
        scales = torch.rand(period, device="cuda", generator=g) * 1e-3 + 1e-4
    dense = codes.double().reshape(N, K)
    if period:
        dense = dense * scales.double()[torch.arange(N * K, device="cuda") % period].reshape(N, K)
    return T.FrozenWeight(codes, T.W_INT8, scales, N, K, period or 1), dense


# (at least 64 rows in every residue class of the flat scale index: the kernel's own condition)
@pytest.mark.parametrize("compute", [T.F32, T.BF16])
@pytest.mark.parametrize("M", [3, 16, 17, 32])
@pytest.mark.parametrize("N,K,period", [(192, 128, 192), (320, 128, 10), (1408, 2048, 1408), (2048, 1408, 2048), (960, 384, 960),
                                        (256, 4096, 256), (208, 3968, 1), (80, 2176, 0),
                                        (1280, 5632, 1280), (640, 14336, 640)])
def test_against_64_bits(N, K, period, M, compute):
    w, dense = _weight(N, K, period, N + K + M)
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.empty(M, K, device="cuda").normal_(0, 1, generator=g).to(T.TORCH_DTYPE[compute])
    y = T.qlinear_forward(x, w, compute, T.F32).double()
    want = x.double() @ dense.t()
    assert ((y - want).norm() / want.norm()).item() <= BOUND


@pytest.mark.parametrize("compute", [T.F32, T.BF16])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_rows_without_numbers(bad, compute):
    w, dense = _weight(512, 2048, 512, 3)
    g = torch.Generator(device="cuda").manual_seed(8)
    x = torch.empty(5, 2048, device="cuda").normal_(0, 1, generator=g).to(T.TORCH_DTYPE[compute])
    x[1, 3] = bad
    x[4, 2047] = bad
    y = T.qlinear_forward(x, w, compute, T.F32)
    finite = torch.isfinite(y)
    assert not finite[1].any() and not finite[4].any() and finite[[0, 2, 3]].all()
    want = x[[0, 2, 3]].double() @ dense.t()
    assert ((y[[0, 2, 3]].double() - want).norm() / want.norm()).item() <= BOUND
