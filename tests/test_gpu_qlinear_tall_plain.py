"""int8 forward with one round of tall tiles (caifx_gemm_tall.hpp without segments), against the CPU oracle's restatement of
CAIF_DeviceFrozenLinear (src/caif_device_frozen_linear.cpp).

Bound: operands bit-identical to the oracle's and fp32 sums in another order: 2e-5 of the largest result, plus half the spacing of
a 16-bit result's values (2^-8 of the value at most in bf16, 2^-11 in fp16)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T                                   # noqa: E402
from gpu_helpers import dev_as, host, make_weight, max_rel_err        # noqa: E402


# the fewest rows; a last row tile of a few rows, and whole tiles; columns that end inside a tile; as many tiles as compute units and fewer;
# scale vectors of 1 to 25 classes
@pytest.mark.parametrize("M,N,K,dt", [(769, 10240, 1280, 2), (801, 9600, 1536, 1), (999, 14336, 1792, 1), (1024, 14336, 2048, 2), (1100, 12288, 1536, 2),
                                      (801, 12800, 1280, 2), (1000, 8192, 8192, 2)])
def test_against_the_oracle(orc, M, N, K, dt):
    rng = np.random.default_rng(M + N + K)
    ow, w = make_weight(orc, rng, N, K, "int8pc")
    x = dev_as(rng.normal(0, 1, (M, K)), dt)
    add = dev_as(rng.normal(0, 1, (M, N)), dt)
    workspace = torch.zeros(2 * N * K, dtype=torch.uint8, device="cuda")
    y32 = host(T.qlinear_forward(x, w, dt, workspace=workspace))
    assert not workspace.any()                                        # no copy of the weight, no partial sums: this kernel
    y16, ya = host(T.qlinear_forward(x, w, dt, dt)), host(T.qlinear_forward(x, w, dt, dt, addend=add))
    rows = np.unique(np.array([0, 15, 16, 127, 128, 255, 256, M // 2, M - 2, M - 1]))
    want = orc.frozen_linear_forward(host(x)[rows], ow, dt)
    half = 2.0 ** -8 if dt == 2 else 2.0 ** -11
    assert max_rel_err(y32[rows], want) <= 2e-5
    assert max_rel_err(y16[rows], want) <= 2e-5 + half
    assert max_rel_err(ya, y16 + host(add)) <= half
    assert np.array_equal(y16, host(torch.from_numpy(y32).to(torch.bfloat16 if dt == 2 else torch.float16)))
    assert np.array_equal(host(T.qlinear_forward(x, w, dt, workspace=torch.empty(0, dtype=torch.uint8, device="cuda"))), y32)
