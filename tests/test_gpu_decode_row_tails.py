"""One and two activation rows through the decode kernels: reductions whose last chunk (2048 codes for int4, 1024 for int8) is
missing, one piece long, one piece short or whole, and every result dtype, against the CPU oracle
(src/caif_device_frozen_linear.cpp:382-524).  int4 and int8 with one scale take the row-linear kernels (caifx_gemv_rowlin.hip);
int8 per channel takes them where the scale vector leaves classes of 256 rows or more, which
test_int8_with_a_scale_vector asks for, and the row-block kernel elsewhere.

Bound: these kernels multiply codes with scales folded in afterwards (or into the activations), the oracle rounds
code * scale to the compute dtype first: 4e-3 of the largest result at bf16, as in test_gpu_qlinear_skinny.py, an eighth of that at
fp16 (three more bits in that rounding); a 16-bit result adds its own, half the spacing of significands of 8 bits (bf16, 2^-8) or
11 (fp16, 2^-11)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T                                  # noqa: E402
from gpu_helpers import dev_as, host, make_weight, max_rel_err        # noqa: E402


@pytest.mark.parametrize("kind", ["int4", "int8pc", "int8pt"])
@pytest.mark.parametrize("K", [128, 1920, 2048, 2176, 3968, 5120, 6144, 8320, 10240, 12160, 14336, 16256])
def test_reduction_tails(orc, kind, K):
    rng = np.random.default_rng(K)
    # int8 per-channel: one class of rows up to K = 2176, eight of 128 rows at K = 3968, 8320, 12160 and 16256 (row-block kernel);
    # N is ragged against the rows of a wave and of a workgroup
    N = {"int4": 1037, "int8pt": 777, "int8pc": K if K <= 2176 else 1024}[kind]
    ow, dw = make_weight(orc, rng, N, K, kind)
    for M in (1, 2):
        for cd, yd in ((2, 0), (2, 2), (1, 1)):
            x = dev_as(rng.normal(0, 1, (M, K)), cd)
            y = T.qlinear_forward(x, dw, cd, yd)
            want = orc.frozen_linear_forward(host(x), ow, cd)
            assert np.isfinite(host(y)).all()
            assert max_rel_err(host(y), want) <= 4e-3 + (2.0 ** -8 if yd == 2 else 0), (M, cd, yd)


def _bound(cd, yd):
    return (4e-3 if cd == 2 else 4e-3 / 8) + {0: 0.0, 1: 2.0 ** -11, 2: 2.0 ** -8}[yd]


@pytest.mark.parametrize("N,K,classes", [(777, 1024, 1), (1030, 1920, 4), (600, 2176, 2), (1100, 3072, 4), (777, 3968, 1), (1040, 4096, 4),
                                         (600, 4224, 2), (1100, 5504, 4), (6160, 6400, 8), (6150, 8176, 2), (1030, 7168, 4), (600, 12288, 2),
                                         (300, 16384, 1), (11010, 11008, 4)])
def test_int8_with_a_scale_vector(orc, N, K, classes):
    # a period of `classes` rows; whole chunks, partial ones with one to four chunks, and beyond K = 4096 in two and four slices
    assert classes * 256 <= N and (K <= 4096 or K % 1024 == 0 or N >= 11008 or (K <= 8192 and (N >= 6144 or K <= 6144)))
    rng = np.random.default_rng(N + K)
    period = classes * K
    codes = rng.integers(-127, 128, N * K).astype(np.int8)
    scales = rng.uniform(1e-4, 2e-4, period).astype(np.float32)
    ow = orc.FrozenWeight(codes, orc.W_INT8, scales, N, K, period, 128)
    dw = T.FrozenWeight(torch.from_numpy(codes).cuda(), T.W_INT8, torch.from_numpy(scales).cuda(), N, K, period, 128)
    for M in (1, 2):
        for cd, xd, yd in ((2, 2, 0), (2, 2, 2), (1, 1, 1), (2, 0, 2), (1, 0, 0)):
            x = dev_as(rng.normal(0, 1, (M, K)), xd)
            want = orc.frozen_linear_forward(host(x), ow, cd)
            assert max_rel_err(host(T.qlinear_forward(x, dw, cd, yd)), want) <= _bound(cd, yd), (M, cd, xd, yd)


@pytest.mark.parametrize("K", [5248, 7168, 8064, 9984])
def test_int4_between_the_chunk_counts(orc, K):
    rng = np.random.default_rng(K)
    ow, dw = make_weight(orc, rng, 1037, K, "int4")
    for M in (1, 2):
        for cd, xd, yd in ((2, 2, 0), (2, 2, 2), (1, 1, 1), (2, 0, 2)):
            x = dev_as(rng.normal(0, 1, (M, K)), xd)
            want = orc.frozen_linear_forward(host(x), ow, cd)
            assert max_rel_err(host(T.qlinear_forward(x, dw, cd, yd)), want) <= _bound(cd, yd), (M, cd, xd, yd)
