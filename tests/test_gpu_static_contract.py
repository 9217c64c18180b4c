"""caifx_qlinear_forward_static against caifx_qlinear_forward on both sides of the dense copy of the weight: the same bits with a
workspace for partial tiles, refused exactly where those exceed the buffer, and the fp32 sums of the larger workspace's call
in another order (2e-5 of the largest result, as between the other matrix-core kernels; int4 codes scaled after the product
against codes rounded to bf16 first: half of 2^-8 per product)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T      # noqa: E402

SCRATCH_BYTES = 8 << 20


@pytest.mark.parametrize("kind", ["int4", "int8"])
@pytest.mark.parametrize("M,N,K", [(64, 2048, 4096), (128, 4096, 4096), (160, 14336, 2048), (512, 4096, 4096), (768, 2048, 2048), (999, 14336, 4096), (2048, 11008, 4096)])
def test_static_is_the_call_with_room_for_partial_tiles(kind, M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M)
    normal = lambda *s: torch.empty(s, device="cuda").normal_(generator=gen)      # noqa: E731
    if kind == "int4":
        p, s = T.quantize_int4_per_group(normal(N, K), 128)
        w = T.FrozenWeight(p, T.W_INT4_GROUP, s, N, K, 1, 128)
    else:
        q, s = T.quantize_int8(normal(K, N), True)
        w = T.FrozenWeight(q.reshape(-1), T.W_INT8, s, N, K, N)
    x = normal(M, K).to(torch.bfloat16)
    sizes = (M, N, K, T.BF16, T.BF16, w.w_kind, 0)
    partials, whole = capi.lib().caifx_qlinear_partials_workspace_bytes(*sizes), capi.lib().caifx_qlinear_workspace_bytes(*sizes)
    assert partials <= whole and partials < 2 * N * K + SCRATCH_BYTES
    y = torch.full((M, N), float("nan"), device="cuda")
    st = capi.lib().caifx_qlinear_forward_static(M, N, K, x.data_ptr(), T.BF16, T.BF16, w.wq.data_ptr(), w.w_kind, w.scales.data_ptr(),
                                                 w.scale_period, w.group_size, y.data_ptr(), T.F32,
                                                 torch.cuda.current_stream().cuda_stream)
    assert (st == 0) == (partials <= SCRATCH_BYTES)
    if st:
        assert "scratch" in capi.status_string(st) and bool(torch.isnan(y).all())
        return
    assert torch.equal(y, T.qlinear_forward(x, w, T.BF16, workspace=torch.empty(partials, dtype=torch.uint8, device="cuda")))
    other = T.qlinear_forward(x, w, T.BF16)
    assert float((y - other).abs().max()) <= (2.0 ** -9 if kind == "int4" else 2e-5) * float(other.abs().max())


@pytest.mark.parametrize("kind", ["int4", "int8"])
def test_gating_in_the_store_is_the_separate_calls_without_a_workspace(kind):
    # long segments, where the separate calls copy the experts' weights if they are given room for it
    gen = torch.Generator(device="cuda").manual_seed(9)
    normal = lambda *s: torch.empty(s, device="cuda").normal_(generator=gen)      # noqa: E731
    E, N, K, rows = 4, 1408, 1024, 8000
    ws = []
    for _ in range(E):
        if kind == "int4":
            p, s = T.quantize_int4_per_group(normal(N, K), 128)
            ws.append(T.FrozenWeight(p, T.W_INT4_GROUP, s, N, K, 1, 128))
        else:
            q, s = T.quantize_int8(normal(K, N), True)
            ws.append(T.FrozenWeight(q.reshape(-1), T.W_INT8, s, N, K, N))
    bank, empty = T.GroupedFrozenWeights(ws), torch.empty(0, dtype=torch.uint8, device="cuda")
    assert capi.lib().caifx_qlinear_grouped_workspace_bytes(E, rows, N, K, T.BF16, T.BF16, bank.w_kind, 0) == 2 * E * N * K
    off = torch.tensor([0, 2100, 2100, 5000, rows], dtype=torch.int32, device="cuda")
    x, gate = normal(rows, K).to(torch.bfloat16), normal(rows, N).to(torch.bfloat16)
    up, hidden = T.qlinear_grouped_forward_swiglu(x, off, bank, gate, T.BF16)
    alone = T.qlinear_grouped_forward(x, off, bank, T.BF16, T.BF16, workspace=empty)
    assert torch.equal(up, alone) and torch.equal(hidden, T.silu_multiply(gate, alone))
