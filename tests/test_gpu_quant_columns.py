"""Per-column int8 quantisation around the edges of its workgroups (256 columns, chunks of 32 to 256 rows whose partial
maxima wait in the codes' memory, 64-row blocks), bit-exact against the oracle (src/caif_cuda_kernels_quant.cu:515-560)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                                  # noqa: E402
from gpu_helpers import dev                                           # noqa: E402


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 31, 32, 33, 63, 65, 257, 1031])
@pytest.mark.parametrize("cols", [3, 4, 8, 252, 256, 260, 1028])
def test_bit_exact(orc, rows, cols):
    rng = np.random.default_rng(rows * 2000 + cols)
    w = rng.normal(0, 0.02, (rows, cols)).astype(np.float32)
    w[:, 0] = 0.0                                      # a column without a maximum: scale 1
    w[rows - 1, cols - 1] = -3.0                        # the maxima of the last row and the last column count
    w[rows // 2, cols // 2] = 2.0
    q, s = T.quantize_int8(dev(w), True)
    qo, so = orc.quantize_int8_per_channel(w)
    assert np.array_equal(s.cpu().numpy(), so) and np.array_equal(q.cpu().numpy(), qo)
    # a source that is not 16-byte aligned takes the element-wise kernels: same bits
    buf = torch.empty(rows * cols + 1, dtype=torch.float32, device="cuda")
    x = buf[1:].reshape(rows, cols)
    x.copy_(dev(w))
    q2, s2 = T.quantize_int8(x, True)
    assert torch.equal(q2, q) and torch.equal(s2, s)


# strips of 32, 16 and 8 columns held by one workgroup: with and without the pieces in LDS, the most rows of each form and one
# more, a last strip that is not full
@pytest.mark.parametrize("rows,cols", [(8, 7000), (768, 7004), (769, 7168), (1024, 7000), (1025, 7004), (1537, 7000), (2048, 7000), (2049, 12288),
                                       (3073, 12292), (4096, 12288), (4097, 12288), (1024, 5000), (1025, 2052), (65, 2052), (2048, 2048), (2049, 36)])
def test_strips(orc, rows, cols):
    rng = np.random.default_rng(rows + cols)
    w = rng.standard_normal((rows, cols), dtype=np.float32)
    w[:, 1] = 0.0
    w[rows - 1, cols - 1], w[0, cols - 2], w[rows // 2, 5] = -9.0, 8.0, 7.0
    q, s = T.quantize_int8(dev(w), True)
    qo, so = orc.quantize_int8_per_channel(w)
    assert np.array_equal(s.cpu().numpy(), so) and np.array_equal(q.cpu().numpy(), qo)


@pytest.mark.parametrize("offset", [4, 8, 12, 1])
@pytest.mark.parametrize("rows,cols", [(8, 4), (65, 260), (1031, 1028), (2100, 260)])
def test_codes_at_any_address(orc, rows, cols, offset):
    # a slice of a packed checkpoint: the partial maxima wait in the codes' memory whatever its alignment
    w = np.random.default_rng(rows + cols).normal(0, 0.02, (rows, cols)).astype(np.float32)
    src, scales = dev(w), torch.empty(cols, device="cuda")
    held = torch.full((rows * cols + 32,), 99, dtype=torch.int8, device="cuda")
    codes = held[offset:offset + rows * cols]
    capi.call("caifx_quantize_int8_per_channel", src.data_ptr(), codes.data_ptr(), scales.data_ptr(), rows, cols,
              torch.cuda.current_stream().cuda_stream)
    qo, so = orc.quantize_int8_per_channel(w)
    assert np.array_equal(codes.cpu().numpy().reshape(rows, cols), qo) and np.array_equal(scales.cpu().numpy(), so)
    assert bool((held[:offset] == 99).all()) and bool((held[offset + rows * cols:] == 99).all())
