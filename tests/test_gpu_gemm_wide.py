"""The large-M path through a dense copy of the weight in the workspace (caifx_gemm_wide.hip): each of its three tile
shapes with partial tiles in both directions, odd and even step counts, every weight kind, forward and input gradient,
every result dtype and the fused addend, against the CPU oracle (src/caif_device_frozen_linear.cpp:382-524, :528-660).
test_the_copy_is_made_and_used holds sizes that the path is chosen for and sees the copy written; the sizes of
test_against_the_oracle lie on both sides of the choice.

Bound: the operands are the oracle's (the weight rounded to the compute type once), the products are summed in fp32 in
another order: 2e-5 of the largest result, as for the other matrix-core kernels; a 16-bit result adds half the spacing of
its values, which for a significand of p bits is 2^-p of the value at most (bf16: p = 8, fp16: p = 11), the addend's
rounding once more."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                             # noqa: E402
from gpu_helpers import dev_as, host, make_weight, max_rel_err        # noqa: E402

ULP = {0: 0.0, 1: 2.0 ** -11, 2: 2.0 ** -8}

# (M, N, K): 256 x 256, 128 x 256 and 128 x 128 tiles, ragged against them; 2, 3 and many 64-deep steps
SHAPES = [(3900, 4040, 128), (2049, 4104, 192), (1160, 3080, 320), (2300, 1920, 448), (1500, 2112, 192), (2500, 1408, 320)]


def _rows(m):
    return np.unique(np.concatenate([np.arange(2), [m // 2, m - 1], np.arange(120, 132), np.arange(250, 260)]))


@pytest.mark.parametrize("kind", ["int4", "int8pc", "int8pt", "int8none", "bf16"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_against_the_oracle(orc, kind, M, N, K):
    rng = np.random.default_rng(M + N + K)
    cd = 2 if kind == "bf16" or (M + K) % 3 else 1
    for backward in (False, True):
        n, k = (K, N // 64 * 64) if backward else (N, K)        # the reduction is K forward, N backward
        if kind == "int4":
            k = max(128, k // 128 * 128)
        if kind == "bf16":
            w = torch.from_numpy(rng.normal(0, 0.02, (n, k)).astype(np.float32)).cuda().to(torch.bfloat16)
            dw = T.FrozenWeight(w.reshape(-1), T.W_BF16, None, n, k)
        else:
            ow, dw = make_weight(orc, rng, n, k, kind)
        R, C = (n, k) if backward else (k, n)
        x = dev_as(rng.normal(0, 1, (M, R)), cd)
        run = T.qlinear_backward_input if backward else T.qlinear_forward
        sel = _rows(M)
        if kind == "bf16":
            want = host(x)[sel].astype(np.float64) @ (host(w).astype(np.float64) if backward else host(w).astype(np.float64).T)
        else:
            want = (orc.frozen_linear_backward if backward else orc.frozen_linear_forward)(host(x)[sel], ow, cd)
        for yd in (0, cd):
            assert max_rel_err(host(run(x, dw, cd, yd))[sel], want) <= 2e-5 + ULP[yd], (backward, yd)
        add = dev_as(rng.normal(0, 1, (M, C)), cd)
        got = host(run(x, dw, cd, cd, addend=add))[sel]
        plain = host(run(x, dw, cd, cd))[sel]
        assert max_rel_err(got, plain + host(add)[sel]) <= ULP[cd], backward      # one rounding of the sum


@pytest.mark.parametrize("kind", ["int4", "int8pc"])
def test_smaller_workspace_falls_back(orc, kind):
    # the dense copy is optional: with less (or no) workspace the kernels that dequantise inside the product run
    rng = np.random.default_rng(5)
    M, N, K = 2048, 2048, 2048
    ow, dw = make_weight(orc, rng, N, K, kind)
    assert capi.lib().caifx_qlinear_workspace_bytes(M, N, K, T.BF16, T.BF16, dw.w_kind, 1) >= 2 * N * K
    x = dev_as(rng.normal(0, 1, (M, N)), 2)
    small = torch.empty(16, dtype=torch.uint8, device="cuda")
    got, want = T.qlinear_backward_input(x, dw, T.BF16, workspace=small), T.qlinear_backward_input(x, dw, T.BF16)
    assert max_rel_err(host(got), host(want)) <= 2e-5


# The smallest products found, by a search over the rule, that the path is chosen for: weight kind, direction, then 256 x 256, 128 x 256
# and 128 x 128 tiles with an even and an odd number of 64-deep steps (int4 forward: whole groups, so even), all ragged
CHOSEN = [("bf16", 0, 3350, 2344, 128), ("bf16", 0, 3212, 2448, 192), ("bf16", 0, 4659, 776, 128), ("bf16", 0, 4101, 912, 192),
          ("bf16", 0, 2478, 536, 128), ("bf16", 0, 529, 2504, 192), ("bf16", 1, 4850, 128, 2184), ("bf16", 1, 3390, 192, 2312),
          ("bf16", 1, 4652, 128, 792), ("bf16", 1, 4136, 192, 912), ("bf16", 1, 4035, 512, 656), ("bf16", 1, 4113, 448, 648),
          ("int4", 0, 4353, 2736, 384), ("int4", 0, 4627, 784, 640), ("int4", 0, 4041, 648, 1408), ("int4", 1, 3095, 384, 3968),
          ("int4", 1, 3217, 320, 3840), ("int4", 1, 1294, 640, 3072), ("int4", 1, 1282, 576, 3072), ("int4", 1, 4744, 1408, 640),
          ("int4", 1, 2964, 1472, 1024), ("int8pc", 0, 4619, 2568, 128), ("int8pc", 0, 3334, 2336, 192), ("int8pc", 0, 1025, 3600, 256),
          ("int8pc", 0, 4712, 776, 320), ("int8pc", 0, 516, 2232, 512), ("int8pc", 0, 2224, 536, 448), ("int8pc", 1, 4372, 128, 2712),
          ("int8pc", 1, 3347, 192, 2312), ("int8pc", 1, 1544, 256, 2472), ("int8pc", 1, 3585, 320, 1032), ("int8pc", 1, 2238, 512, 536),
          ("int8pc", 1, 1157, 448, 1048), ("int8pt", 1, 3347, 192, 2312), ("int8none", 0, 4619, 2568, 128)]


@pytest.mark.parametrize("kind,backward,M,N,K", CHOSEN)
def test_the_copy_is_made_and_used(orc, kind, backward, M, N, K):
    rng = np.random.default_rng(M + N + K)
    cd = 1 if kind != "bf16" and M % 2 else 2
    R, C = (N, K) if backward else (K, N)
    x = dev_as(rng.normal(0, 1, (M, R)), cd)
    sel = _rows(M)
    if kind == "bf16":
        w = dev_as(rng.normal(0, 0.02, (N, K)), 2)
        dw = T.FrozenWeight(w.reshape(-1), T.W_BF16, None, N, K)
        want = host(x)[sel].astype(np.float64) @ (host(w).astype(np.float64) if backward else host(w).astype(np.float64).T)
    else:
        ow, dw = make_weight(orc, rng, N, K, kind)
        want = (orc.frozen_linear_backward if backward else orc.frozen_linear_forward)(host(x)[sel], ow, cd)
    run = T.qlinear_backward_input if backward else T.qlinear_forward
    for yd in (0, cd):
        workspace = torch.zeros(2 * N * K, dtype=torch.uint8, device="cuda")
        assert max_rel_err(host(run(x, dw, cd, yd, workspace=workspace))[sel], want) <= 2e-5 + ULP[yd], yd
        if kind != "bf16" or backward:
            assert bool(workspace[-1024:].any())              # (a stored 16-bit weight is used as it is in the forward)
    add = dev_as(rng.normal(0, 1, (M, C)), cd)
    plain = host(run(x, dw, cd, cd))[sel]
    assert max_rel_err(host(run(x, dw, cd, cd, addend=add))[sel], plain + host(add)[sel]) <= ULP[cd]


@pytest.mark.parametrize("kind", ["int4", "int8pc"])
def test_replays_of_a_captured_step(orc, kind):
    # the copy and the product of both directions in one graph: every replay, with new inputs in the captured buffers and eager
    # work in between, gives the eager call's bits
    rng = np.random.default_rng(77)
    M, N, K = 2049, 4096, 4096
    _, dw = make_weight(orc, rng, N, K, kind)
    x, dy = (torch.empty(M, n, device="cuda", dtype=torch.bfloat16) for n in (K, N))
    a, b = (torch.empty(M, n, device="cuda", dtype=torch.bfloat16) for n in (N, K))
    step = lambda: (T.qlinear_forward(x, dw, T.BF16, T.BF16, addend=a), T.qlinear_backward_input(dy, dw, T.BF16, T.BF16, addend=b))      # noqa: E731
    fill = lambda: [t.normal_() for t in (x, dy, a, b)]      # noqa: E731
    fill()
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for _ in range(4):
        fill()
        graph.replay()
        want = step()
        torch.cuda.synchronize()
        assert all(torch.equal(g, w) for g, w in zip(got, want))
