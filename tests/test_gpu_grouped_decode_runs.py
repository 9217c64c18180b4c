"""Few rows per expert: the list of weight blocks cut into equal runs, one per workgroup.  Against the quantised weights in 64
bits, for runs that end inside a unit, span experts, classes and passes, cover one block or none, and more than 64 experts."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi                # noqa: E402
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


def _fresh(backward, x, offsets, gw, compute, out_dtype, shift, addend=None):
    """caifx_qlinear_grouped_fresh into memory that holds NaN, `shift` elements past a 16-byte boundary; nothing in front of the result and
    behind it may change."""
    rows, cols = x.shape[0], gw.K if backward else gw.N
    guard = 64
    whole = torch.full((guard + shift + rows * cols + guard,), float("nan"), device="cuda", dtype=T.TORCH_DTYPE[out_dtype])
    y = whole[guard + shift:guard + shift + rows * cols]
    ws = torch.empty(16 << 20, device="cuda", dtype=torch.uint8)
    capi.call("caifx_qlinear_grouped_fresh", int(backward), len(gw.weights), offsets.data_ptr(), rows, gw.N, gw.K, x.data_ptr(), T.CODE_OF[x.dtype],
              compute, gw.wq_ptrs.data_ptr(), gw.w_kind, gw.scales_ptrs.data_ptr(), gw.scale_period, gw.group_size, y.data_ptr(), out_dtype,
              0 if addend is None else addend.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert torch.isnan(whole[:guard + shift]).all() and torch.isnan(whole[guard + shift + rows * cols:]).all()
    return y.reshape(rows, cols)


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
    y = _fresh(False, x, offsets, gw, T.BF16, T.F32, 0)
    assert rows + 2 <= 16 * E      # the kernel this is about
    assert not y[rows:].any()
    lo = 0
    for e, n in enumerate(counts):
        if n:
            want = x[lo:lo + n].double() @ dense[e].t()
            assert ((y[lo:lo + n].double() - want).norm() / want.norm()).item() <= BOUND[kind], (e, n)
        lo += n


OFFSETS = [([0, 3, 7], 7), ([2, 3, 9], 14), ([0, 0, 0], 5), ([5, 5, 5], 9), ([5, 8, 2, 4], 11), ([-4, 6, 99], 8), ([4, 2, 6], 9), ([3] + [4] * 70, 6)]


def _covered(offsets, rows):
    c = torch.zeros(rows, dtype=torch.bool, device="cuda")
    for lo, hi in zip(offsets, offsets[1:]):
        lo = min(max(lo, 0), rows)
        c[lo:max(lo, min(max(hi, 0), rows))] = True
    return c


# offsets out of range or order lose rows and leave the others zero; byte ranges that begin and end off a 16-byte boundary
@pytest.mark.parametrize("kind", ["int8", "int4"])
@pytest.mark.parametrize("shift", [0, 1, 8])
@pytest.mark.parametrize("offsets,rows", OFFSETS)
def test_rows_outside_the_segments(kind, shift, offsets, rows):
    E, N, K = len(offsets) - 1, 192, 128
    gw, dense = _bank(kind, E, N, K, 3)
    x = torch.empty(rows, K, device="cuda").normal_(0, 1, generator=torch.Generator(device="cuda").manual_seed(1)).to(torch.bfloat16)
    off = torch.tensor(offsets, device="cuda", dtype=torch.int32)
    assert rows <= 16 * E      # the decode kernel: cleared by the product's own launch
    want = torch.zeros(rows, N, device="cuda", dtype=torch.bfloat16)
    T.qlinear_grouped_forward(x, off, gw, T.BF16, T.BF16, out=want)       # into a result that is cleared already
    assert torch.equal(_fresh(False, x, off, gw, T.BF16, T.BF16, shift), want)
    assert torch.equal(T.qlinear_grouped_forward(x, off, gw, T.BF16, T.BF16), want)
    covered = _covered(offsets, rows)
    assert not want[~covered].any() and want[covered].any(dim=1).all()


# the tiled kernel: the gradient with an addend and without, and a forward of more rows than the decode kernel takes (the other grouped
# kernels, and offsets out of order, in test_gpu_grouped_clearing.py)
@pytest.mark.parametrize("kind", ["int8", "int4"])
@pytest.mark.parametrize("form", ["gradient", "addend", "forward"])
@pytest.mark.parametrize("offsets,rows", [([2, 30, 41], 50), ([0, 33, 40], 40), ([5, 5, 5], 40)])
def test_rows_outside_the_segments_in_other_paths(kind, form, offsets, rows):
    N, K = 192, 128
    gw, dense = _bank(kind, 2, N, K, 3)
    back = form != "forward"
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.empty(rows, N if back else K, device="cuda").normal_(0, 1, generator=gen).to(torch.bfloat16)
    add = torch.empty(rows, K, device="cuda").normal_(0, 1, generator=gen).to(torch.bfloat16) if form == "addend" else None
    off = torch.tensor(offsets, device="cuda", dtype=torch.int32)
    want = torch.zeros(rows, K if back else N, device="cuda", dtype=torch.bfloat16)
    if back:
        T.qlinear_grouped_backward_input(x, off, gw, T.BF16, T.BF16, out=want, addend=add)
    else:
        T.qlinear_grouped_forward(x, off, gw, T.BF16, T.BF16, out=want)
    got = _fresh(back, x, off, gw, T.BF16, T.BF16, 0, add)
    covered = _covered(offsets, rows)
    assert torch.equal(got, want) and not got[~covered].any() and got[covered].any(dim=1).all()
