"""fp32 compute over int8 and int4 codes on the 16-bit matrix cores (operands as bf16 pieces), forward and input gradient, against
the weight (fp32 code * scale) in 64 bits: each of the three tiles, with the reduction shared and not, at row counts on the edges of 16-row
blocks and of tiles, ragged columns, one step and many, scale vectors that wrap inside a step.  The plan that the host makes is asked for
with each case, so that a case is on the tile that it names.  (Values out of the pieces' range: test_gpu_fp32_pieces_range.py.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T      # noqa: E402


def _bound(R):
    # six products per 32 reduction elements enter an fp32 sum, each rounded to 2^-24 of it; the products left out are below 2^-25
    return 2.0 ** -24 * ((6 * R / 32) ** 0.5 + 1)


def _weight(kind, N, K, gen):
    if kind == "int4":
        p, s = T.quantize_int4_per_group(torch.empty(N, K, device="cuda").normal_(0, 0.02, generator=gen), 128)
        return T.FrozenWeight(p, T.W_INT4_GROUP, s, N, K, 1, 128), T.dequantize_int4_per_group(p, s, N * K, 128).double().reshape(N, K)
    period = {"channel": N, "wrap": 68, "one": 1, "none": 0}[kind]
    codes = torch.randint(-128, 128, (N * K,), device="cuda", generator=gen, dtype=torch.int8)
    w, scales = codes.float(), None
    if period:
        scales = torch.rand(period, device="cuda", generator=gen) * 1e-3 + 1e-4
        w = w * scales[torch.arange(N * K, device="cuda") % period]
    return T.FrozenWeight(codes, T.W_INT8, scales, N, K, period or 1), w.double().reshape(N, K)


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


KINDS = ["int4", "channel", "wrap", "one", "none"]
NO_LIMIT = 2 ** 63
# rows of a tile, reduction shared, M, columns, reduction (of the forward: N, K; of the gradient: K, N)
CASES = [(32, False, 33, 80, 64), (32, False, 65, 2064, 192), (32, True, 33, 80, 320), (32, True, 95, 1104, 704), (32, True, 129, 208, 1088),
         (64, False, 513, 4112, 64), (64, False, 2095, 1040, 64), (64, True, 33, 4112, 704), (64, True, 600, 1040, 704), (64, True, 2100, 80, 704),
         (128, False, 513, 6160, 64), (128, False, 1151, 3088, 64), (128, False, 513, 6160, 320), (128, False, 200, 14352, 192)]
INT8_CASES = [(128, True, 65, 8208, 704), (128, True, 4100, 80, 1088)]


def _both_ways(kind, M, C, R):
    gen = torch.Generator(device="cuda").manual_seed(M + C + R)
    w, dense = _weight(kind, C, R, gen)
    x = torch.empty(M, R, device="cuda").normal_(0, 1, generator=gen)
    assert _rel(T.qlinear_forward(x, w, T.F32), x.double() @ dense.t()) <= _bound(R)
    w, dense = _weight(kind, R, C, gen)
    dy = torch.empty(M, R, device="cuda").normal_(0, 1e-3, generator=gen)
    assert _rel(T.qlinear_backward_input(dy, w, T.F32), dy.double() @ dense) <= _bound(R)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("bm,shared,M,C,R", CASES)
def test_every_tile(pieces_plans, kind, bm, shared, M, C, R):
    plan = pieces_plans([(M, C, R, int(kind == "int4"), NO_LIMIT)])[0]
    assert plan[0] == bm and (plan[1] > 1) == shared and not plan[4], plan
    _both_ways(kind, M, C, R)


@pytest.mark.parametrize("kind", KINDS[1:])
@pytest.mark.parametrize("bm,shared,M,C,R", INT8_CASES)
def test_every_tile_int8(pieces_plans, kind, bm, shared, M, C, R):
    plan = pieces_plans([(M, C, R, 0, NO_LIMIT)])[0]
    assert plan[0] == bm and (plan[1] > 1) == shared and not plan[4], plan
    _both_ways(kind, M, C, R)


# rows around the tiles' edges, whichever kernel the host chooses, with the workspace and without
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("M", [33, 48, 64, 65, 81, 128, 129, 200])
@pytest.mark.parametrize("N,K", [(64, 64), (192, 320), (1344, 2048)])
def test_forward_and_gradient(kind, M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    w, dense = _weight(kind, N, K, gen)
    x = torch.empty(M, K, device="cuda").normal_(0, 1, generator=gen)
    dy = torch.empty(M, N, device="cuda").normal_(0, 1e-3, generator=gen)
    empty = torch.empty(0, dtype=torch.uint8, device="cuda")
    for ws in (None, empty):
        assert _rel(T.qlinear_forward(x, w, T.F32, workspace=ws), x.double() @ dense.t()) <= _bound(K)
        assert _rel(T.qlinear_backward_input(dy, w, T.F32, workspace=ws), dy.double() @ dense) <= _bound(N)


@pytest.mark.parametrize("M", [2, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(192, 192), (4096, 4096), (80, 192)])
def test_few_rows_int4(M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M)
    w, dense = _weight("int4", N, K, gen)
    x = torch.empty(M, K, device="cuda").normal_(0, 1, generator=gen)
    assert _rel(T.qlinear_forward(x, w, T.F32), x.double() @ dense.t()) <= _bound(K)


# 16-bit activations on each tile; results of another type are the fp32 results rounded
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("out", [T.F32, T.BF16, T.F16])
@pytest.mark.parametrize("kind,bm,M,C,R", [("channel", 32, 100, 208, 320), ("int4", 32, 100, 208, 320), ("channel", 64, 600, 1040, 704),
                                           ("int4", 64, 600, 1040, 704), ("channel", 128, 513, 6160, 64), ("int4", 128, 513, 6160, 64)])
def test_types(pieces_plans, kind, bm, M, C, R, dtype, out):
    plan = pieces_plans([(M, C, R, int(kind == "int4"), NO_LIMIT)])[0]
    assert plan[0] == bm and not plan[4]
    gen = torch.Generator(device="cuda").manual_seed(1)
    w, dense = _weight(kind, C, R, gen)
    x = torch.empty(M, R, device="cuda").normal_(0, 1, generator=gen).to(dtype)
    y = T.qlinear_forward(x, w, T.F32, out)
    assert torch.equal(y, T.qlinear_forward(x, w, T.F32, T.F32).to(T.TORCH_DTYPE[out]))
    assert _rel(T.qlinear_forward(x, w, T.F32), x.double() @ dense.t()) <= _bound(R)
    w, dense = _weight(kind, R, C, gen)
    dx = T.qlinear_backward_input(x, w, T.F32, out)
    assert torch.equal(dx, T.qlinear_backward_input(x, w, T.F32, T.F32).to(T.TORCH_DTYPE[out]))
    assert _rel(T.qlinear_backward_input(x, w, T.F32), x.double() @ dense) <= _bound(R)


def test_extreme_values(pieces_plans):
    # codes without zeros, so that an infinity times a weight is one
    N, K, M = 128, 320, 40
    assert not pieces_plans([(M, N, K, 0, NO_LIMIT)])[0][4]
    codes = torch.randint(1, 128, (N * K,), device="cuda", dtype=torch.int8)
    w = T.FrozenWeight(codes, T.W_INT8, torch.full((1,), 2.0 ** -8, device="cuda"), N, K, 1)
    x = torch.zeros(M, K, device="cuda")
    big, tiny = 3.4028234e38, 2.0 ** -100
    x[0, 3], x[1, 5], x[2, 7], x[3, 9], x[4, 11] = big, -big, float("inf"), float("-inf"), float("nan")
    x[5, 200] = tiny
    x[6, 100] = torch.tensor(0x7f800001, dtype=torch.int32).view(torch.float32)          # a NaN that truncation would make an infinity
    y = T.qlinear_forward(x, w, T.F32)
    dense = codes.double().reshape(N, K) * 2.0 ** -8
    want = x.double()[[0, 1, 5]] @ dense.t()
    assert torch.allclose(y[[0, 1, 5]].double(), want, rtol=2.0 ** -22, atol=0)
    assert (y[2] == float("inf")).all() and (y[3] == float("-inf")).all() and torch.isnan(y[4]).all() and torch.isnan(y[6]).all()
    assert not y[7:].any()
