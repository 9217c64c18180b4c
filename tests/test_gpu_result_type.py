"""A 16-bit result has the bits of the fp32 result rounded once (the caller's `.To(StorageT)` after the layer,
src/caif_device_moe_frozen_expert.cpp:119-126): the result's type may not choose a kernel with other sums.  One size for every
kernel: one and two rows with whole and partial last chunks, row blocks, shared reductions, each large-M path."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T                       # noqa: E402

SIZES = [(1, 1024, 2048), (1, 4096, 2176), (1, 1037, 4096), (1, 2048, 6400), (1, 4096, 11008), (1, 1024, 14336), (2, 4096, 3968), (2, 1000, 7168),
         (5, 2048, 4096), (16, 1024, 8192), (24, 2048, 2048), (64, 2048, 2048), (100, 4096, 4096), (320, 8192, 1024), (999, 4096, 2048),
         (2048, 11008, 4096), (2049, 4104, 192)]


@pytest.mark.parametrize("kind", ["int4", "int8pc", "int8pt", "bf16"])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_16_bit_results_are_the_fp32_results_rounded(kind, M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    normal = lambda *s: torch.empty(s, device="cuda").normal_(generator=gen)      # noqa: E731
    cd = T.F16 if K == 6400 and kind != "bf16" else T.BF16
    if kind == "bf16":
        w = T.FrozenWeight(normal(N, K).to(torch.bfloat16).reshape(-1), T.W_BF16, None, N, K)
    elif kind == "int4":
        K = max(K // 128 * 128, 128)
        p, s = T.quantize_int4_per_group(normal(N, K), 128)
        w = T.FrozenWeight(p, T.W_INT4_GROUP, s, N, K, 1, 128)
    else:
        q, s = T.quantize_int8(normal(K, N), kind == "int8pc")
        w = T.FrozenWeight(q.reshape(-1), T.W_INT8, s, N, K, N if kind == "int8pc" else 1)
    for run, R in ((T.qlinear_forward, K), (T.qlinear_backward_input, N)):
        x = normal(M, R).to(T.TORCH_DTYPE[cd])
        assert torch.equal(run(x, w, cd, cd), run(x, w, cd, T.F32).to(T.TORCH_DTYPE[cd])), run.__name__
