"""Rows that no segment covers, cleared by the launch of each 16-bit grouped kernel: into memory that holds NaN, with offsets out of range or
order; and the search for a tile of equal height among more than 64 experts."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                                     # noqa: E402
from test_gpu_grouped_decode_runs import _bank, _covered, _fresh              # noqa: E402


def _one_scale(E, N, K):
    g = torch.Generator(device="cuda").manual_seed(E)
    weights = []
    for _ in range(E):
        q, s = T.quantize_int8(torch.empty(K, N, device="cuda").normal_(0, 0.02, generator=g), per_channel=False)
        weights.append(T.FrozenWeight(q.reshape(-1), T.W_INT8, s, N, K, 1))
    return T.GroupedFrozenWeights(weights)


def _offsets(rows):
    """Four segments of which the last three may step down, begin late, end early or run past the buffer; none covers another's rows."""
    u = rows // 16
    return [[0, 3 * u, 3 * u, 9 * u, rows], [3, u, 4 * u + 1, 9 * u, rows - 5], [5, 5, 5, 5, 5], [11 * u, 14 * u + 1, 2 * u, 4 * u, 4 * u],
            [-4, 6 * u, 6 * u, 9 * u + 1, rows + 99], [4 * u, 2 * u, 6 * u, 6 * u, 9 * u]]


# the kernel that takes the call: tall tiles (int8, a scale vector), the int8 forward with one scale, dense copies of the weights (long
# segments; the size query says so), the tiled kernel
@pytest.mark.parametrize("which", range(6))
@pytest.mark.parametrize("kernel,kind,N,K,rows,back,addend", [
    ("tall", "int8", 320, 256, 1500, False, False), ("tall", "int8", 384, 256, 1500, True, False), ("tall", "int8", 384, 256, 1500, True, True),
    ("one scale", None, 512, 256, 8200, False, False),
    ("copies", "int8", 1024, 1024, 12100, False, False), ("copies", "int4", 1024, 1024, 12100, True, True),
    ("tiled", "int4", 256, 256, 700, False, False), ("tiled", "int8", 192, 128, 700, True, False), ("tiled", "int4", 192, 128, 700, True, True)])
def test_rows_outside_the_segments(kernel, kind, N, K, rows, back, addend, which):
    offsets = _offsets(rows)[which]
    gw = _bank(kind, 4, N, K, 3)[0] if kind else _one_scale(4, N, K)
    need = capi.lib().caifx_qlinear_grouped_workspace_bytes(4, rows, N, K, T.BF16, T.BF16, gw.w_kind, int(back))
    assert need == (8 * N * K if kernel == "copies" else 0)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.empty(rows, N if back else K, device="cuda").normal_(0, 1, generator=gen).to(torch.bfloat16)
    add = torch.empty(rows, K, device="cuda").normal_(0, 1, generator=gen).to(torch.bfloat16) if addend else None
    off = torch.tensor(offsets, device="cuda", dtype=torch.int32)
    want = torch.zeros(rows, K if back else N, device="cuda", dtype=torch.bfloat16)
    if back:
        T.qlinear_grouped_backward_input(x, off, gw, T.BF16, T.BF16, out=want, addend=add)      # into a result that is cleared already
    else:
        T.qlinear_grouped_forward(x, off, gw, T.BF16, T.BF16, out=want)
    got = _fresh(back, x, off, gw, T.BF16, T.BF16, 0, add)
    covered = _covered(offsets, rows)
    assert torch.equal(got, want) and not got[~covered].any() and got[covered].any(dim=1).all()


# Bound: 256 or 384 products of operands that are the same, their fp32 sums in another order: sqrt(384) roundings of 2^-24 as a random walk,
# 1.2e-6 of the result's 2-norm; twice that.
@pytest.mark.parametrize("back", [False, True])
@pytest.mark.parametrize("counts", [[20, 0, 97, 1, 300, 64, 31, 129, 0, 257] * 7, [0] * 130 + [2113, 0, 33], [65] * 64 + [700]])
def test_many_experts(counts, back):
    E, N, K, first = len(counts), 384, 256, 2
    gw, dense = _bank("int8", E, N, K, E)
    bounds = torch.tensor([first] + counts).cumsum(0).tolist()
    rows = bounds[-1] + 3
    assert rows > 16 * E      # not the decode kernel, whose weights are not rounded
    x = torch.empty(rows, N if back else K, device="cuda").normal_(0, 1, generator=torch.Generator(device="cuda").manual_seed(5)).to(torch.bfloat16)
    got = _fresh(back, x, torch.tensor(bounds, device="cuda", dtype=torch.int32), gw, T.BF16, T.F32, 0)
    assert not got[:first].any() and not got[bounds[-1]:].any()
    for e, (lo, hi) in enumerate(zip(bounds, bounds[1:])):
        if lo < hi:
            w = dense[e].float().to(torch.bfloat16).double()
            want = x[lo:hi].double() @ (w if back else w.t().contiguous())
            assert ((got[lo:hi].double() - want).norm() / want.norm()).item() <= 2.4e-6, e
