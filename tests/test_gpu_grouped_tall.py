"""Grouped forward and input gradient in tiles of up to 256 rows (caifx_gemm_tall.hpp), against the CPU oracle's per-expert
restatement of CAIF_DeviceMoEFrozenExpert (src/caif_device_moe_frozen_expert.cpp:92-332).

Bound: as in test_gpu_grouped_wide.py, operands bit-identical to the oracle's and fp32 sums in another order: 2e-5 of the
largest result, plus half the spacing of a 16-bit result's values (2^-8 of the value at most in bf16, 2^-11 in fp16)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                             # noqa: E402
from gpu_helpers import dev, dev_as, host, make_weight, max_rel_err   # noqa: E402

# rows on and around the edges of a 16-row operand tile, of the instantiated heights (64, 96 .. 256) and of the cut into equal
# tiles; empty segments between them
ROWS = [1, 0, 31, 64, 65, 96, 97, 128, 0, 129, 160, 191, 192, 225, 255, 256, 257, 385, 513, 2]


# thirty segments of about 240 rows, too many for two tiles each at a time: tiles of 224 and 256 rows
HIGH = [224 + 7 * i % 33 for i in range(30)] + [257, 193]


@pytest.mark.parametrize("rows,N,K,dt", [
    (ROWS, 1408, 2048, 2),     # eleven classes of weight rows with the same scales; a column tile with idle waves (forward)
    (HIGH, 1408, 2048, 2),
    (ROWS, 2048, 1408, 2),     # sixteen classes, idle waves in the gradient
    (ROWS, 256, 256, 2),       # one class, the shortest reduction
    (ROWS, 2176, 256, 1),      # seventeen classes, the most whose table holds neighbouring rows
    (ROWS, 2304, 384, 2),      # six classes
    (ROWS, 1984, 256, 2),      # 31 classes in the forward; its gradient's reduction is no multiple of 128
    (ROWS, 384, 1152, 1),
])
def test_segments(orc, rows, N, K, dt):
    rng = np.random.default_rng(N + K)
    E, first = len(rows), 3
    offsets = (first + np.concatenate([[0], np.cumsum(rows)])).astype(np.int32)
    total = int(offsets[-1]) + 2
    pairs = [make_weight(orc, rng, N, K, "int8pc") for _ in range(E)]
    ows, gw = [p[0] for p in pairs], T.GroupedFrozenWeights([p[1] for p in pairs])
    off = dev(offsets)
    x, dy = dev_as(rng.normal(0, 1, (total, K)), dt), dev_as(rng.normal(0, 1e-2, (total, N)), dt)
    add = dev_as(rng.normal(0, 1e-2, (total, K)), dt)
    if rows is HIGH:      # the tiles under test are those that run
        stamps = torch.zeros(4 * 4096, dtype=torch.int64, device="cuda")
        capi.lib().caifx_qlinear_grouped_tile_stamps(stamps.data_ptr(), 4096)
        T.qlinear_grouped_forward(x, off, gw, dt, dt)
        torch.cuda.synchronize()
        capi.lib().caifx_qlinear_grouped_tile_stamps(None, 0)
        heights = stamps.view(-1, 4)[:, 1] & 0xFFFFFFFF
        assert 224 < int(heights.max()) <= 256
    y32, dx32 = (host(f(a, off, gw, dt)) for f, a in ((T.qlinear_grouped_forward, x), (T.qlinear_grouped_backward_input, dy)))
    y16, dx16 = (host(f(a, off, gw, dt, dt)) for f, a in ((T.qlinear_grouped_forward, x), (T.qlinear_grouped_backward_input, dy)))
    dxa = host(T.qlinear_grouped_backward_input(dy, off, gw, dt, dt, addend=add))
    dxa32 = host(T.qlinear_grouped_backward_input(dy, off, gw, dt, addend=add.float()))
    for r in (y32, dx32, y16, dx16, dxa):
        assert not r[:first].any() and not r[offsets[-1]:].any()      # rows outside the segments: zero
    half = 2.0 ** -8 if dt == 2 else 2.0 ** -11
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if lo == hi:
            continue
        sel = np.unique(np.clip(np.concatenate([lo + np.arange(0, hi - lo, 61), lo + 32 * np.arange(9), lo + 32 * np.arange(9) - 1,
                                                [(lo + hi) // 2, hi - 1]]), lo, hi - 1))
        want, dwant = (orc.frozen_linear_forward(host(x)[sel], ows[e], dt), orc.frozen_linear_backward(host(dy)[sel], ows[e], dt))
        assert max_rel_err(y32[sel], want) <= 2e-5 and max_rel_err(dx32[sel], dwant) <= 2e-5, e
        assert max_rel_err(y16[sel], want) <= 2e-5 + half and max_rel_err(dx16[sel], dwant) <= 2e-5 + half, e
        assert max_rel_err(dxa[sel], dx16[sel] + host(add)[sel]) <= half, e
        assert max_rel_err(dxa32[sel], dx32[sel] + host(add)[sel]) <= 2.0 ** -23, e


def test_gating_in_the_store():
    # the up projection and the down projection's gradient with the gating in their stores: the bits of the separate launches
    gen = torch.Generator(device="cuda").manual_seed(4)
    normal = lambda *s: torch.empty(s, device="cuda").normal_(generator=gen)      # noqa: E731
    E, H, D = 5, 640, 512

    def bank(n, k):
        ws = []
        for _ in range(E):
            q, s = T.quantize_int8(normal(k, n), True)
            ws.append(T.FrozenWeight(q.reshape(-1), T.W_INT8, s, n, k, n))
        return T.GroupedFrozenWeights(ws)
    up_w, down_w = bank(H, D), bank(D, H)
    off = torch.tensor([0, 130, 130, 131, 700, 998], dtype=torch.int32, device="cuda")
    for dt in (torch.bfloat16, torch.float16):
        code = T.BF16 if dt == torch.bfloat16 else T.F16
        x, gate, dy = normal(1000, D).to(dt), normal(1000, H).to(dt), normal(1000, D).to(dt)
        up, hidden = T.qlinear_grouped_forward_swiglu(x, off, up_w, gate, code)
        want = T.qlinear_grouped_forward(x, off, up_w, code, code)
        assert torch.equal(up[:998], want[:998]) and torch.equal(hidden[:998], T.silu_multiply(gate, want)[:998])
        assert not hidden[998:].any()
        gg, gu = T.qlinear_grouped_backward_input_swiglu(dy, off, down_w, gate, up, code)
        wg, wu = T.swiglu_backward(gate, up, T.qlinear_grouped_backward_input(dy, off, down_w, code, code))
        assert torch.equal(gg[:998], wg[:998]) and torch.equal(gu[:998], wu[:998])
