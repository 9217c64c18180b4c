"""Few rows per expert: the list of weight blocks cut into equal runs, one per workgroup.  Against the quantised weights in 64
bits, for runs that end inside a unit, span experts, classes and passes, cover one block or none, and more than 64 experts."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T      # noqa: E402

# int8: the digits' share, as in the row-block kernel's own test.  int4: the sums run over code + 136 (rms 136 against 2.9 of the
# codes alone) before the offset's share is taken off, so their fp32 roundings, 2^-24 each and about eight in a row, weigh 47
# times as much: 47 * 2^-24 * sqrt(8) = 7.9e-6; twice that.
BOUND = {"int8": 4.5e-6, "int4": 1.6e-5}


def _bank(kind, E, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    weights, dense = [], []
    for _ in range(E):
        w = torch.empty(N, K, device="cuda").normal_(0, 0.02, generator=g)
        if kind == "int4":
            p, s = T.quantize_int4_per_group(w, 128)
            weights.append(T.FrozenWeight(p, T.W_INT4_GROUP, s, N, K, 1, 128))
            dense.append(T.dequantize_int4_per_group(p, s, N * K, 128).double().reshape(N, K))
        else:
            q, s = T.quantize_int8(w.reshape(K, N), per_channel=True)
            weights.append(T.FrozenWeight(q.reshape(-1), T.W_INT8, s, N, K, N))
            dense.append((q.reshape(-1).double() * s.double()[torch.arange(N * K, device="cuda") % N]).reshape(N, K))
    return T.GroupedFrozenWeights(weights), dense


@pytest.mark.parametrize("kind", ["int8", "int4"])
@pytest.mark.parametrize("N,K", [(1408, 512), (192, 128), (64, 2176)])
@pytest.mark.parametrize("counts", [[1], [0, 0, 3], [16, 0, 17, 1, 33, 2, 0, 5], [2] * 33, [1, 0] * 35 + [40, 0, 3],
                                    [0] * 130 + [7, 1]])
def test_runs(kind, N, K, counts):
    E = len(counts)
    gw, dense = _bank(kind, E, N, K, N + K + E)
    offsets = torch.tensor([0] + counts, device="cuda").cumsum(0).to(torch.int32)
    rows = int(sum(counts))
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.empty(rows + 2, K, device="cuda").normal_(0, 1, generator=g).to(torch.bfloat16)
    y = T.qlinear_grouped_forward(x, offsets, gw, T.BF16, T.F32)
    assert rows + 2 <= 16 * E or len(counts) < 8      # the kernel this is about
    assert not y[rows:].any()
    lo = 0
    for e, n in enumerate(counts):
        if n:
            want = x[lo:lo + n].double() @ dense[e].t()
            bound = BOUND[kind] if rows + 2 <= 16 * E else 3e-3          # the tiled kernel rounds code * scale to bf16
            assert ((y[lo:lo + n].double() - want).norm() / want.norm()).item() <= bound, (e, n)
        lo += n


@pytest.mark.parametrize("kind", ["int8", "int4"])
@pytest.mark.parametrize("offsets,rows", [([0, 3, 7], 7), ([2, 3, 9], 14), ([0, 0, 0], 5), ([5, 5, 5], 9), ([5, 8, 2, 4], 11), ([-4, 6, 99], 8),
                                          ([4, 2, 6], 9), ([3] + [4] * 70, 6)])
def test_rows_outside_the_segments(kind, offsets, rows):
    # cleared by the product's own launch; offsets out of range or order lose rows and leave the others zero
    E, N, K = len(offsets) - 1, 192, 128
    gw, dense = _bank(kind, E, N, K, 3)
    x = torch.empty(rows, K, device="cuda").normal_(0, 1, generator=torch.Generator(device="cuda").manual_seed(1)).to(torch.bfloat16)
    off = torch.tensor(offsets, device="cuda", dtype=torch.int32)
    want = torch.zeros(rows, N, device="cuda", dtype=torch.bfloat16)
    T.qlinear_grouped_forward(x, off, gw, T.BF16, T.BF16, out=want)       # into a result that is cleared already
    dirty = torch.full((rows, N), float("nan"), device="cuda", dtype=torch.bfloat16)      # what a fresh result's memory may hold
    del dirty
    assert torch.equal(T.qlinear_grouped_forward(x, off, gw, T.BF16, T.BF16), want)
    covered = torch.zeros(rows, dtype=torch.bool)
    for e in range(E):
        lo = min(max(offsets[e], 0), rows)
        covered[lo:max(lo, min(max(offsets[e + 1], 0), rows))] = True
    assert not want[~covered.cuda()].any()
