"""Clearing of the rows of a grouped result that no segment covers (caifx_qlinear_grouped_zero_rest), byte for byte."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi      # noqa: E402


@pytest.mark.parametrize("offsets,rows,cols,dtype", [([0, 3, 7], 7, 5, torch.bfloat16), ([2, 3, 4], 9, 5, torch.bfloat16), ([0, 0], 3, 1, torch.bfloat16),
                                                     ([1, 1, 1], 3000, 1027, torch.float32), ([5, 8, 2], 11, 8, torch.bfloat16), ([-4, 6, 99], 8, 3, torch.float32)])
def test_zero_rest(offsets, rows, cols, dtype):
    # byte ranges that start and end off a 16-byte boundary, nothing to clear, everything, entries out of range or order
    y = torch.ones(rows + 2, cols, device="cuda", dtype=dtype)
    off = torch.tensor(offsets, device="cuda", dtype=torch.int32)
    capi.call("caifx_qlinear_grouped_zero_rest", len(offsets) - 1, off.data_ptr(), rows, cols * y.element_size(), y[1:].data_ptr(),
              torch.cuda.current_stream().cuda_stream)
    lo, hi = (min(max(v, 0), rows) for v in (offsets[0], offsets[-1]))
    want = torch.ones_like(y)
    want[1:1 + lo] = 0
    want[1 + max(lo, hi):1 + rows] = 0
    assert torch.equal(y, want)
