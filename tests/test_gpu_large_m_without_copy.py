"""The tests of the kernels that dequantise inside the product, run without room for a dense copy of the weight: with it many of
their sizes go to caifx_gemm_wide.hip, which test_gpu_gemm_wide.py covers.  These kernels are what the static entry point, the
C++ layer and callers with a smaller workspace run on.  Same assertions and bounds as in the modules they come from."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from caif_amd import capi, torch_ops as T                             # noqa: E402
import test_gpu_qlinear_gemm as tiled                                 # noqa: E402
import test_gpu_qlinear_gemm_int4_dx as int4_dx                       # noqa: E402
import test_gpu_qlinear_gemm_int4_fwd as int4_fwd                     # noqa: E402
import test_gpu_qlinear_gemm_int8_fwd as int8_fwd                     # noqa: E402


@pytest.fixture(autouse=True)
def room_for_partial_tiles_only(monkeypatch):
    def limited(run, backward):
        def call(x, fw, compute_dtype, y_dtype=T.F32, out=None, workspace=None, addend=None):
            if workspace is None:
                M = x.numel() // (fw.N if backward else fw.K)
                n = capi.lib().caifx_qlinear_partials_workspace_bytes(M, fw.N, fw.K, T.CODE_OF[x.dtype], compute_dtype, fw.w_kind, backward)
                assert n < 2 * fw.N * fw.K or M <= 512          # too little for the copy, or too few rows for one
                workspace = torch.empty(n, dtype=torch.uint8, device="cuda")
            return run(x, fw, compute_dtype, y_dtype, out, workspace, addend)
        return call
    monkeypatch.setattr(T, "qlinear_forward", limited(T.qlinear_forward, 0))
    monkeypatch.setattr(T, "qlinear_backward_input", limited(T.qlinear_backward_input, 1))


def _take(module, *names):
    for name in names:
        globals()[f"{name}_{module.__name__[len('test_gpu_qlinear_'):]}"] = getattr(module, name)


_take(tiled, "test_single_tile_and_multi_tile", "test_ragged_tiles", "test_dtype_mixes", "test_int4_group_sizes",
      "test_config3_prefill_shapes_sampled_rows", "test_fused_output_cast", "test_linearity_and_adjoint_at_full_size")
_take(int8_fwd, "test_per_channel_full_tiles", "test_one_scale_and_no_scale", "test_last_row_tile_runs_over_its_row_blocks_only",
      "test_ragged_columns", "test_compute_and_result_types", "test_fused_add_equals_cast_then_add",
      "test_one_hot_rows_return_single_weight_columns", "test_repeat_calls_are_bit_identical")
_take(int4_dx, "test_full_tiles", "test_ragged_rows", "test_compute_and_result_types", "test_fused_add_equals_cast_then_add",
      "test_one_hot_rows_return_single_weight_rows", "test_adjoint_with_the_forward")
_take(int4_fwd, "test_full_tiles", "test_ragged_rows_and_columns", "test_compute_and_result_types",
      "test_fused_add_equals_cast_then_add", "test_one_hot_rows_return_single_weight_columns", "test_repeat_calls_are_bit_identical")
