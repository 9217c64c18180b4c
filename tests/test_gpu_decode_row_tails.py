"""One and two activation rows through the row-linear decode kernels (caifx_gemv_rowlin.hip): reductions whose last chunk
(2048 codes for int4, 1024 for int8) is missing, one piece long, one piece short or whole, every chunk count of the
fixed-shape kernels, and every result dtype, against the CPU oracle (src/caif_device_frozen_linear.cpp:382-524).

Bound: these kernels multiply codes with scales folded in afterwards (or into the activations), the oracle rounds
code * scale to the compute dtype first: 4e-3 of the largest result at bf16, as in test_gpu_qlinear_skinny.py; a 16-bit
bf16 result adds its own rounding, half the spacing of 8-bit significands (2^-8)."""
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
    # int8 per-channel: a period that leaves 1 or few residue classes, so that the row-linear kernel is taken; N is
    # ragged against the rows of a wave and of a workgroup
    N = {"int4": 1037, "int8pt": 777, "int8pc": K if K <= 2176 else 1024}[kind]
    ow, dw = make_weight(orc, rng, N, K, kind)
    for M in (1, 2):
        for cd, yd in ((2, 0), (2, 2), (1, 1)):
            x = dev_as(rng.normal(0, 1, (M, K)), cd)
            y = T.qlinear_forward(x, dw, cd, yd)
            want = orc.frozen_linear_forward(host(x), ow, cd)
            assert np.isfinite(host(y)).all()
            assert max_rel_err(host(y), want) <= 4e-3 + (2.0 ** -8 if yd == 2 else 0), (M, cd, yd)
