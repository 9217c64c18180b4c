"""Forward whose tiles all run at once, on the kernel whose waves split the reduction (caifx_gemm_few.hip), against the CPU
oracle's restatement of CAIF_DeviceFrozenLinear (src/caif_device_frozen_linear.cpp).

Bound: operands bit-identical to the oracle's and fp32 sums in another order: 2e-5 of the largest result, plus half the spacing of
a 16-bit result's values (2^-8 of the value at most in bf16, 2^-11 in fp16)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                             # noqa: E402
from gpu_helpers import dev_as, host, make_weight, max_rel_err        # noqa: E402


BLOCKS = {33: 2, 48: 2, 65: 2, 96: 2, 40: 3, 60: 4, 75: 5, 90: 6, 100: 7, 150: 5, 220: 7, 130: 2, 200: 2, 700: 2}


# tiles of two to seven 16-row blocks, and the last of several that begins before its own rows; columns that end inside a 64-column
# tile; reductions of fewer units than waves, of an odd number per wave, shared among workgroups or not.  Groups of 32 are the tiled
# kernel's: what it gives beside this one.  The workspace has room for shared reductions and none for a copy of the weight, so that the plan
# is what runs, and holds the sums of the plan's parts and nothing else.
@pytest.mark.parametrize("kind,group", [("int4", 128), ("int4", 32), ("int8pc", 128), ("int8pt", 128), ("int8", 128)])
@pytest.mark.parametrize("M,N,K,dt", [(33, 512, 512, 2), (48, 64, 512, 1), (65, 200, 1152, 2), (96, 512, 4096, 2), (40, 8448, 640, 2), (60, 8448, 640, 1),
                                      (75, 8456, 640, 2), (90, 8448, 512, 2), (100, 8448, 640, 2), (150, 8192, 640, 1), (220, 8192, 512, 2),
                                      (130, 1024, 1024, 2), (200, 448, 3200, 2), (700, 320, 2176, 2)])
def test_against_the_oracle(orc, few_plans, kind, group, M, N, K, dt):
    rng = np.random.default_rng(M + N + K)
    ow, w = make_weight(orc, rng, N, K, kind, group=group)
    x = dev_as(rng.normal(0, 1, (M, K)), dt)
    add = dev_as(rng.normal(0, 1, (M, N)), dt)
    room = capi.lib().caifx_qlinear_partials_workspace_bytes(M, N, K, dt, dt, w.w_kind, 0)
    workspace = torch.zeros(room + 4096, dtype=torch.uint8, device="cuda")
    y32 = host(T.qlinear_forward(x, w, dt, workspace=workspace[:room]))
    if group == 128:
        (_, blocks, parts, _), = few_plans([(M, N, K, {"int4": 0, "int8pc": 1}.get(kind, 2))])
        assert parts > 0 and blocks == BLOCKS[M], (blocks, parts)
        used = parts * M * N * 4 if parts > 1 else 0
        assert used <= room and not workspace[used:].any() and (used == 0 or bool(workspace[used - 4096:used].any()))
    y16 = host(T.qlinear_forward(x, w, dt, dt, workspace=workspace[:room]))
    ya = host(T.qlinear_forward(x, w, dt, dt, addend=add, workspace=workspace[:room]))
    rows = np.unique(np.concatenate([np.arange(0, M, 13), [15, 16, 31, 32, M // 2, M - 2, M - 1]]))
    want = orc.frozen_linear_forward(host(x)[rows], ow, dt)
    half = 2.0 ** -8 if dt == 2 else 2.0 ** -11
    assert max_rel_err(y32[rows], want) <= 2e-5
    assert max_rel_err(y16[rows], want) <= 2e-5 + half
    assert max_rel_err(ya, y16 + host(add)) <= half
    assert np.array_equal(y16, host(torch.from_numpy(y32).to(torch.bfloat16 if dt == 2 else torch.float16)))
