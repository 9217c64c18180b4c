"""Which calls ask for a dense copy of the weight in the workspace (csrc/caifx_gemm_wide.hip).  The sizes are ones where one
of the two ways was measured at least 5 % faster than the other on an MI355X; the size query needs no GPU."""
import pytest

from caif_amd import capi

INT8, INT4, BF16_W, BF16 = capi.W_INT8, capi.W_INT4_GROUP, capi.W_BF16, 2


def _copies(M, N, K, kind, backward):
    return capi.lib().caifx_qlinear_workspace_bytes(M, N, K, BF16, BF16, kind, backward) >= 2 * N * K


@pytest.mark.parametrize("kind,backward,M,N,K", [
    (INT4, 0, 256, 14336, 4096), (INT4, 0, 192, 14336, 2048),
    (INT4, 0, 320, 8192, 1024), (INT4, 0, 384, 11008, 4096), (INT4, 0, 768, 5952, 2048), (INT4, 0, 1536, 8192, 1024), (INT4, 1, 256, 4096, 14336), (INT4, 1, 512, 4096, 14336),
    (BF16_W, 1, 160, 4096, 14336), (BF16_W, 1, 512, 4096, 14336), (BF16_W, 1, 1024, 14336, 4096)])
def test_a_copy_used_for_few_rows_is_not_made(kind, backward, M, N, K):
    assert not _copies(M, N, K, kind, backward)


@pytest.mark.parametrize("kind,backward,M,N,K", [
    (INT8, 0, 160, 14336, 4096), (INT8, 0, 768, 14336, 4096), (INT8, 0, 999, 14336, 4096), (INT8, 0, 320, 11008, 4096),
    (INT8, 1, 768, 14336, 4096), (INT8, 0, 512, 4096, 4096), (INT8, 0, 2048, 2048, 2048), (INT8, 1, 2048, 8192, 1024),
    (INT4, 0, 2048, 11008, 4096), (INT4, 0, 1024, 11008, 4096), (INT4, 1, 768, 4096, 4096), (INT4, 1, 4096, 11008, 4096),
    (BF16_W, 1, 1536, 14336, 4096), (BF16_W, 1, 1024, 8192, 4096), (BF16_W, 1, 768, 4096, 4096),
    # one scale: the tiled kernel takes twice as long, so the query, which does not know the scales, counts the copy
    (INT8, 0, 64, 14336, 4096), (INT8, 1, 64, 4096, 14336)])
def test_a_copy_that_pays_is_made(kind, backward, M, N, K):
    assert _copies(M, N, K, kind, backward)


def test_reductions_longer_than_a_grid_of_the_transposing_pass():
    assert _copies(8192, (1 << 22) - 64, 512, INT8, 1) and not _copies(8192, 1 << 22, 512, INT8, 1)


def _grouped_copies(E, rows, N, K, kind, backward):
    return capi.lib().caifx_qlinear_grouped_workspace_bytes(E, rows, N, K, BF16, BF16, kind, backward) == 2 * E * N * K


@pytest.mark.parametrize("kind,backward,E,rows,N,K,copies", [
    (INT8, 0, 33, 29700, 1024, 1536, False), (INT8, 0, 33, 36300, 1024, 1536, False), (INT4, 1, 16, 14400, 512, 2048, False),
    (INT4, 0, 8, 16000, 512, 1024, False), (INT8, 0, 64, 48640, 512, 512, False),
    (INT8, 0, 8, 24576, 1408, 2048, True), (INT4, 1, 8, 24576, 1408, 2048, True), (INT4, 0, 16, 24576, 1408, 2048, True),
    (INT8, 1, 8, 12800, 1408, 2048, True), (INT8, 0, 8, 24576, 512, 1024, True)])
def test_expert_segments(kind, backward, E, rows, N, K, copies):
    assert _grouped_copies(E, rows, N, K, kind, backward) == copies
