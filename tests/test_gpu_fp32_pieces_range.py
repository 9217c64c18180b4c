"""fp32 compute over int8 and int4 codes as products of bf16 pieces: values that no bf16 pieces hold (infinities, NaN, numbers too
large or too small, and products past the largest fp32 number) run on the fp32 instruction, step by step.  Against the same values in
64 bits rounded to fp32, one such value a row, placed in different steps, waves and parts of the reduction."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import torch_ops as T      # noqa: E402

INF, NAN = float("inf"), float("nan")
# the activation next to a scale: passes of the largest number by the product alone (2.99e38 * 3000, 1.003e30 * 1e12), in a first
# piece alone (3.4028234e38 rounds to an infinity in bf16), infinities against infinities and against weights that bf16 rounds to
# zero, numbers whose last piece bf16 would cut off (3.7e-36), a NaN that truncation would make an infinity
VALUES = [(2.99e38, 30.0), (-2.99e38, 30.0), (1.003e30, 1e10), (3.4028234e38, 2.0 ** -8), (-3.4028234e38, 2.0 ** -8), (INF, INF), (-INF, INF),
          (1.0, INF), (0.0, INF), (INF, 2.0 ** -145), (INF, 2.0 ** -8), (-INF, 2.0 ** -8), (NAN, 1.0), (1.0, NAN), (3.7e-36, 0.0117), (1.7e-36, 0.5), (2.0 ** -100, 2.0 ** -8),
          (1.1e-33, 1.3e-5), (1.2345678, 1.2345678e-13), (1.2345678e-19, 1.2345678e-11), (1.2345678e15, 1.2345678e15), (0.0, 0.0), (5.0, 0.0), (INF, 0.0), (NAN, 0.0), (2.0 ** -100, 0.0)]


def _expected(x, dense):
    return (x.double() @ dense).float()


def _check(got, want):
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    ok = ~torch.isnan(want)
    inf = torch.isinf(want) & ok
    assert torch.equal(got[inf], want[inf]) and torch.equal(torch.isinf(got) & ok, inf)
    # one product a sum: the fp32 rounding of code * scale, and the product's
    fin = ok & ~inf
    assert torch.allclose(got[fin].double(), want[fin].double(), rtol=2.0 ** -22, atol=0)


def _on_the_pieces(pieces_plans, *calls):
    assert not any(split for *_, split in pieces_plans([(*c, 2 ** 63) for c in calls]))


def _x(M, R, value, gen):
    # row m holds the value at one place; the other rows are left zero
    x = torch.zeros(M, R, device="cuda")
    for i, m in enumerate(range(0, M, 7)):
        x[m, (i * 71 + 13) % R] = value
    return x


@pytest.mark.parametrize("form", ["one", "vector"])
@pytest.mark.parametrize("value,scale", VALUES)
@pytest.mark.parametrize("M,N,K", [(40, 192, 320), (100, 320, 192), (200, 1024, 2048)])
def test_int8(pieces_plans, form, value, scale, M, N, K):
    _on_the_pieces(pieces_plans, (M, N, K, 0), (M, K, N, 0))
    gen = torch.Generator(device="cuda").manual_seed(M)
    codes = torch.randint(-128, 128, (N, K), device="cuda", generator=gen, dtype=torch.int8)
    codes = torch.where(codes == 0, torch.ones_like(codes), codes)          # (zeros against infinities: test_int4)
    if form == "one":
        scales = torch.full((1,), scale, device="cuda")
    else:
        scales = torch.full((N,), 0.25, device="cuda")
        scales[::3] = scale
    dense = (codes.reshape(-1).float() * scales[torch.arange(N * K, device="cuda") % scales.numel()]).double().reshape(N, K)
    w = T.FrozenWeight(codes.reshape(-1), T.W_INT8, scales, N, K, scales.numel())
    for ws in (None, torch.empty(0, dtype=torch.uint8, device="cuda")):
        x = _x(M, K, value, gen)
        _check(T.qlinear_forward(x, w, T.F32, workspace=ws), _expected(x, dense.t()))
        dy = _x(M, N, value, gen)
        _check(T.qlinear_backward_input(dy, w, T.F32, workspace=ws), _expected(dy, dense))


@pytest.mark.parametrize("value,scale", [(1.0, INF), (INF, INF), (-1.5, INF), (1.0, NAN), (INF, 6e-8), (2.99e38, 3000.0), (3.7e-36, 0.0117), (1.0, 6e-8),
                                         (INF, 0.25), (0.0, 0.25)])
@pytest.mark.parametrize("M,N,K", [(40, 192, 320), (100, 320, 192), (200, 1024, 2048)])
def test_int4(pieces_plans, value, scale, M, N, K):
    _on_the_pieces(pieces_plans, (M, N, K, 1), (M, K, N, 1))
    gen = torch.Generator(device="cuda").manual_seed(M)
    packed = torch.randint(0, 256, (N * K // 2,), device="cuda", generator=gen, dtype=torch.uint8)
    scales = torch.full((N * K // 64,), 0.25, device="cuda", dtype=torch.float16)
    scales[::5] = scale
    lo, hi = (packed & 15).to(torch.int32), (packed >> 4).to(torch.int32)
    codes = torch.stack([lo, hi], 1).reshape(-1)
    codes = torch.where(codes > 7, codes - 16, codes)
    dense = (codes.float() * scales.float().repeat_interleave(64)).double().reshape(N, K)
    w = T.FrozenWeight(packed, T.W_INT4_GROUP, scales, N, K, 1, 64)
    x = _x(M, K, value, gen)
    _check(T.qlinear_forward(x, w, T.F32), _expected(x, dense.t()))
    dy = _x(M, N, value, gen)
    _check(T.qlinear_backward_input(dy, w, T.F32), _expected(dy, dense))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("value", [INF, -INF, NAN, 2.0 ** -24, 65504.0])
def test_16_bit_activations(dtype, value):
    gen = torch.Generator(device="cuda").manual_seed(3)
    M, N, K = 100, 192, 320
    codes = torch.randint(1, 128, (N, K), device="cuda", generator=gen, dtype=torch.int8)
    w = T.FrozenWeight(codes.reshape(-1), T.W_INT8, torch.full((1,), 0.037, device="cuda"), N, K, 1)
    dense = (codes.float() * 0.037).double()
    x = _x(M, K, value, gen).to(dtype)
    _check(T.qlinear_forward(x, w, T.F32), _expected(x, dense.t()))


def test_a_step_with_such_a_value_keeps_the_others():
    # every 5th row tiny in one step, the others ordinary: the steps on either side and the rest of the tile keep their results
    gen = torch.Generator(device="cuda").manual_seed(4)
    M, N, K = 130, 320, 704
    codes = torch.randint(-128, 128, (N, K), device="cuda", generator=gen, dtype=torch.int8)
    scales = torch.rand(N, device="cuda", generator=gen) * 1e-3 + 1e-4
    dense = (codes.reshape(-1).float() * scales[torch.arange(N * K, device="cuda") % N]).double().reshape(N, K)
    w = T.FrozenWeight(codes.reshape(-1), T.W_INT8, scales, N, K, N)
    x = torch.empty(M, K, device="cuda").normal_(0, 1, generator=gen)
    x[::5, 200] = 1e-30
    x[::5, 650] = 1e-30
    y, want = T.qlinear_forward(x, w, T.F32).double(), x.double() @ dense.t()
    assert ((y - want).norm() / want.norm()).item() <= 2.0 ** -24 * ((6 * K / 32) ** 0.5 + 1)


@pytest.mark.parametrize("kind", ["int8", "int4"])
@pytest.mark.parametrize("value", [1.0, INF, 3e38])
@pytest.mark.parametrize("M,N,K", [(100, 192, 320), (200, 1024, 2048)])
def test_infinite_weights_without_zeros(kind, value, M, N, K):
    # every operand positive, so that a sum with an infinite term is an infinity and no NaN
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, dy = torch.ones(M, K, device="cuda"), torch.ones(M, N, device="cuda")
    x[::3, K - 70] = value
    dy[::3, 70] = value
    if kind == "int8":
        codes = torch.randint(1, 128, (N * K,), device="cuda", generator=gen, dtype=torch.int8)
        scales = torch.full((N,), 2.0 ** -8, device="cuda")
        scales[70] = INF
        dense = codes.float() * scales[torch.arange(N * K, device="cuda") % N]
        w = T.FrozenWeight(codes, T.W_INT8, scales, N, K, N)
    else:
        codes = torch.randint(1, 8, (N * K,), device="cuda", generator=gen, dtype=torch.uint8)
        scales = torch.full((N * K // 64,), 2.0 ** -8, device="cuda", dtype=torch.float16)
        scales[11] = INF
        dense = codes.float() * scales.float().repeat_interleave(64)
        w = T.FrozenWeight(codes[::2] | codes[1::2] << 4, T.W_INT4_GROUP, scales, N, K, 1, 64)
    dense = dense.double().reshape(N, K)
    for got, want in ((T.qlinear_forward(x, w, T.F32), _expected(x, dense.t())), (T.qlinear_backward_input(dy, w, T.F32), _expected(dy, dense))):
        assert torch.equal(torch.isinf(got), torch.isinf(want)) and not torch.isnan(got).any() and (got > 0).all()
        assert torch.allclose(got, want, rtol=2.0 ** -20, atol=0)
