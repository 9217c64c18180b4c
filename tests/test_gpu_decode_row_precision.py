"""What the one-row decode kernels (caifx_gemv_rowlin.hip) keep of their operands, on values where losing it shows."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T                                  # noqa: E402
from gpu_helpers import dev, dev_as, host, max_rel_err               # noqa: E402


@pytest.mark.parametrize("K", [1024, 2048, 3072, 4096, 5120, 11264, 14336, 16384, 3968, 5504])
@pytest.mark.parametrize("period", [1, 0])
def test_int8_digits_reach_2_to_the_minus_21_of_the_largest_activation(K, period):
    # One activation of 1 meets a code of 0 in every row and each lane's unit is set by others like it; the rest are odd
    # multiples of 2^-21, which digits of 2^-21 or finer hold exactly: what is left is the fp32 sum of at most 16384
    # terms in a tree (2^-20 of the largest result), and a 16-bit result's rounding (half the spacing of 8-bit significands, 2^-8).
    # Partial last chunks beyond K = 6144 need more rows than these for the kernel to be chosen.
    rng = np.random.default_rng(K)
    N = 1500                            # one residue class of 256 rows or more: the row-linear kernels are taken
    codes = rng.integers(-127, 128, (N, K)).astype(np.int8)
    x = rng.choice([-3, -1, 1, 3], K) * 2.0 ** -21
    x[::16] = 1.0                       # every lane's piece of 16 has one
    codes[:, ::16] = 0
    scales = dev(np.ones(1 if period == 1 else K, np.float32))
    w = T.FrozenWeight(dev(codes).reshape(-1), T.W_INT8, scales, N, K, 1 if period == 1 else K)
    want = codes.astype(np.float64) @ x
    xd = dev_as(x[None], 2)
    for yd in (T.F32, T.BF16):
        got = host(T.qlinear_forward(xd, w, T.BF16, yd))[0]
        assert max_rel_err(got, want) <= 2.0 ** -20 + (2.0 ** -8 if yd == T.BF16 else 0), yd


@pytest.mark.parametrize("cd", [T.BF16, T.F16])
@pytest.mark.parametrize("K", [256, 2048, 2304, 3840, 4096, 6144, 6400, 8192, 10240, 12288, 14336, 16384])
def test_int4_groups_of_128_and_of_256_give_the_same_bits(orc, K, cd):
    # The same codes and scales as groups of 256 (the kernel for any group size) and of 128 (the fixed-shape kernels, also
    # with a partial last chunk where the result has 16 bits): the same sums in the same order, so the same bits.
    rng = np.random.default_rng(K)
    N = 1037
    p, s = orc.quantize_to_int4(rng.normal(0, 0.02, (N, K)).astype(np.float32), 256)
    s = s.view(np.float16)
    wide = T.FrozenWeight(dev(p), T.W_INT4_GROUP, dev(s), N, K, 1, 256)
    narrow = T.FrozenWeight(dev(p), T.W_INT4_GROUP, dev(np.repeat(s, 2)), N, K, 1, 128)
    for M in (1, 2) if K <= 14336 else (1,):
        x = dev_as(rng.normal(0, 1, (M, K)), cd)
        for yd in (T.F32, cd):
            assert torch.equal(T.qlinear_forward(x, wide, cd, yd), T.qlinear_forward(x, narrow, cd, yd)), (M, yd)


def _int8(rng, N, K, period):
    codes = rng.integers(-127, 128, (N, K)).astype(np.int8)
    scales = rng.uniform(1e-4, 2e-4, period).astype(np.float32)
    w = T.FrozenWeight(dev(codes).reshape(-1), T.W_INT8, dev(scales), N, K, period)
    return codes * scales[np.arange(N * K) % period].reshape(N, K).astype(np.float64), w


@pytest.mark.parametrize("yd", [T.F32, T.BF16])
@pytest.mark.parametrize("N,K,period", [(777, 1024, 1), (1408, 2176, 1), (1000, 3072, 3072), (2048, 3968, 496), (768, 4096, 4096)])
def test_int8_infinities_come_out_as_the_products_give_them(N, K, period, yd):
    rng = np.random.default_rng(N + K)
    w64, w = _int8(rng, N, K, period)
    for values in ({5: np.inf}, {K - 1: -np.inf}, {0: np.inf, K // 2: np.inf}, {7: np.nan}):
        x = rng.normal(0, 1, (1, K)).astype(np.float32)
        for k, v in values.items():
            x[0, k] = v
        for xd in (T.BF16, T.F32):
            got = host(T.qlinear_forward(dev_as(x, xd), w, T.BF16, yd))[0]
            with np.errstate(invalid="ignore"):
                want = (x[0].astype(np.float64) * w64).sum(axis=1)
            assert not np.isfinite(want).any() and np.array_equal(got, want, equal_nan=True), (values, xd)


@pytest.mark.parametrize("N,K,period", [(777, 1024, 1), (1408, 2176, 1), (2048, 3968, 496)])
def test_int8_activations_near_the_end_of_the_exponent_range(N, K, period):
    # 2^-100 times ordinary values: the same results times 2^-100, to the rounding of code * scale to bf16 (2^-9 each, 4e-3 of the
    # largest result as for the other decode kernels) and the result's own
    rng = np.random.default_rng(K)
    w64, w = _int8(rng, N, K, period)
    x = dev_as(rng.normal(0, 1, (1, K)), 2)
    want = w64 @ host(x)[0].astype(np.float64)
    for shift in (-80, -100, -108):
        got = host(T.qlinear_forward(x * 2.0 ** shift, w, T.BF16, T.BF16))[0].astype(np.float64) * 2.0 ** -shift
        assert max_rel_err(got, want) <= 4e-3 + 2.0 ** -8, shift
