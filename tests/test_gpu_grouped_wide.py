"""Grouped forward and input gradient through dense copies of the experts' weights (caifx_gemm_wide.hip, long segments),
against the CPU oracle's per-expert restatement of
CAIF_DeviceMoEFrozenExpert (src/caif_device_moe_frozen_expert.cpp:92-332).

Bound: as in test_gpu_gemm_wide.py, operands bit-identical to the oracle's and fp32 sums in another order: 2e-5 of the
largest result, plus half the spacing of a 16-bit result's values (bf16: 2^-8 of the value at most)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                             # noqa: E402
from gpu_helpers import dev, dev_as, host, make_weight, max_rel_err   # noqa: E402


def _bank(orc, rng, E, N, K, kind):
    pairs = [make_weight(orc, rng, N, K, kind) for _ in range(E)]
    return [p[0] for p in pairs], T.GroupedFrozenWeights([p[1] for p in pairs])


# 256 x 256, 128 x 256 and 128 x 128 tiles; segments that are empty, of one row, on and around the edges of a tile; rows
# in front of the first segment and behind the last
@pytest.mark.parametrize("kind", ["int8pc", "int4", "int8pt"])
@pytest.mark.parametrize("first,counts,N,K", [(0, [4097, 0, 3500], 1408, 1024), (5, [1, 8191, 256, 5000], 1088, 1152),
                                              (0, [2303, 127, 8011], 1024, 512)])
def test_long_segments(orc, kind, first, counts, N, K):
    rng = np.random.default_rng(N + K)
    E = len(counts)
    offsets = (first + np.concatenate([[0], np.cumsum(counts)])).astype(np.int32)
    total = int(offsets[-1]) + 3
    ows, gw = _bank(orc, rng, E, N, K, kind)
    need = capi.lib().caifx_qlinear_grouped_workspace_bytes(E, total, N, K, T.BF16, T.BF16, gw.w_kind, 1)
    assert need == 2 * E * N * K                                      # the path under test is the one that runs
    off = dev(offsets)
    x, dy = dev_as(rng.normal(0, 1, (total, K)), 2), dev_as(rng.normal(0, 1e-2, (total, N)), 2)
    add = dev_as(rng.normal(0, 1e-2, (total, K)), 2)
    y32, dx32 = (host(f(a, off, gw, T.BF16)) for f, a in ((T.qlinear_grouped_forward, x), (T.qlinear_grouped_backward_input, dy)))
    y16, dx16 = (host(f(a, off, gw, T.BF16, T.BF16)) for f, a in ((T.qlinear_grouped_forward, x), (T.qlinear_grouped_backward_input, dy)))
    dxa = host(T.qlinear_grouped_backward_input(dy, off, gw, T.BF16, T.BF16, addend=add))
    for r in (y32, dx32, y16, dx16, dxa):
        assert not r[:first].any() and not r[offsets[-1]:].any()      # rows outside the segments: zero
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if lo == hi:
            continue
        sel = np.unique(np.clip(np.concatenate([[lo, lo + 127, lo + 128, lo + 255, lo + 256, (lo + hi) // 2], np.arange(hi - 4, hi)]), lo, hi - 1))
        xs, dys = host(x)[sel], host(dy)[sel]
        want, dwant = orc.frozen_linear_forward(xs, ows[e], 2), orc.frozen_linear_backward(dys, ows[e], 2)
        assert max_rel_err(y32[sel], want) <= 2e-5 and max_rel_err(dx32[sel], dwant) <= 2e-5, e
        assert max_rel_err(y16[sel], want) <= 2e-5 + 2.0 ** -8 and max_rel_err(dx16[sel], dwant) <= 2e-5 + 2.0 ** -8, e
        assert max_rel_err(dxa[sel], dx16[sel] + host(add)[sel]) <= 2.0 ** -8, e
