"""fp32 compute over int8 and int4 codes on the 16-bit matrix cores (operands as bf16 pieces), forward and input gradient, against
the weight (fp32 code * scale) in 64 bits: row counts at the edges of 16-row blocks and of the three tiles, ragged columns, one
step and many, shared reductions and none, scale vectors that wrap inside a step, extreme values."""
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


@pytest.mark.parametrize("kind", ["int4", "channel", "wrap", "one", "none"])
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
@pytest.mark.parametrize("N,K", [(192, 192), (4096, 4096), (80, 128)])
def test_few_rows_int4(M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M)
    w, dense = _weight("int4", N, K, gen)
    x = torch.empty(M, K, device="cuda").normal_(0, 1, generator=gen)
    assert _rel(T.qlinear_forward(x, w, T.F32), x.double() @ dense.t()) <= _bound(K)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("out", [T.F32, T.BF16, T.F16])
def test_types(dtype, out):
    gen = torch.Generator(device="cuda").manual_seed(1)
    w, dense = _weight("channel", 256, 512, gen)
    x = torch.empty(100, 512, device="cuda").normal_(0, 1, generator=gen).to(dtype)
    y = T.qlinear_forward(x, w, T.F32, out)
    assert torch.equal(y, T.qlinear_forward(x, w, T.F32, T.F32).to(T.TORCH_DTYPE[out]))
    assert _rel(T.qlinear_forward(x, w, T.F32), x.double() @ dense.t()) <= _bound(512)


def test_extreme_values():
    # codes without zeros, so that an infinity times a weight is one
    N, K, M = 128, 256, 40
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
