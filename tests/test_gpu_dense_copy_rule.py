"""int8 calls whose scales decide whether the weight is copied (csrc/caifx_gemm_wide.hip): the workspace query does not know
them, the call does.  The copy fills the workspace to its last byte; the partial tiles of a shared reduction end far before."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T      # noqa: E402


# measured on an MI355X, copy against no copy: a scale per channel 52 / 47, 55 / 47, 83 / 75, 83 / 73 us; one scale 52 / 93, 54 / 95,
# 82 / 74 (the kernel with a scale table), 82 / 187
@pytest.mark.parametrize("M,N,K,backward,per_channel,copies", [
    (64, 14336, 4096, 0, True, False), (64, 4096, 14336, 1, True, False), (512, 14336, 4096, 0, True, False), (512, 4096, 14336, 1, True, False),
    (64, 14336, 4096, 0, False, True), (64, 4096, 14336, 1, False, True), (512, 14336, 4096, 0, False, False), (512, 4096, 14336, 1, False, True),
    (768, 14336, 4096, 0, True, True)])
def test_the_scales_decide(M, N, K, backward, per_channel, copies):
    gen = torch.Generator(device="cuda").manual_seed(M)
    normal = lambda *s: torch.empty(s, device="cuda").normal_(generator=gen)      # noqa: E731
    codes, scales = T.quantize_int8(normal(K, N), per_channel)
    w = T.FrozenWeight(codes.reshape(-1), T.W_INT8, scales, N, K, N if per_channel else 1)
    x = normal(M, N if backward else K).to(torch.bfloat16)
    run = T.qlinear_backward_input if backward else T.qlinear_forward
    workspace = torch.zeros(2 * N * K, dtype=torch.uint8, device="cuda")
    run(x, w, T.BF16, workspace=workspace)
    assert bool(workspace[-4096:].any()) == copies


def test_a_full_card_does_without_the_copy():
    # the copy is 128 MB more than the call needs: where they cannot be had the call runs on the kernels without it
    # tensors made in place, without larger temporaries: blocks they left behind would have room for the copy
    gen = torch.Generator(device="cuda").manual_seed(3)
    M, N, K = 2048, 8192, 8192
    torch.cuda.empty_cache()
    codes = torch.randint(-127, 128, (N * K,), device="cuda", dtype=torch.int8, generator=gen)
    scales = torch.full((N,), 1e-3, device="cuda")
    w = T.FrozenWeight(codes, T.W_INT8, scales, N, K, N)
    x = torch.empty(M, N, device="cuda", dtype=torch.bfloat16).normal_(generator=gen)
    out = torch.empty(M, K, device="cuda", dtype=torch.bfloat16)
    want = T.qlinear_backward_input(x, w, T.BF16, T.BF16, workspace=torch.empty(0, dtype=torch.uint8, device="cuda"))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (32 << 20)) / total)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(2 * N * K, dtype=torch.uint8, device="cuda")
        assert torch.equal(T.qlinear_backward_input(x, w, T.BF16, T.BF16, out=out), want)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
