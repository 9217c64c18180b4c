"""Size query of the row-block decode kernel.  caifx_qlinear_forward_static takes a call if its partial sums fit the library's own
buffer: which calls it takes is fixed by the slices that the query has always counted (the longest reduction a workgroup covers; half
of it for int8 with few columns), so lengths added to the choice since must not carry a call over the line in either direction."""
import itertools

import pytest

from caif_amd import capi

F32, F16, BF16, INT8, INT4 = 0, 1, 2, 0, 1
LIMIT = 8 << 20


def _counted(M, N, K, compute, kind):
    if compute == F32 and kind == INT4:
        return 0
    reach = 4096 if M <= 16 else 2048
    length = reach
    if M <= 16 and kind == INT8 and N <= (32768 if compute == F32 else 8192):
        length = reach // 2
    slices = -(-K // length)
    if slices > 64:
        slices = -(-K // reach)
    return slices * M * N * 4 if 2 <= slices <= 64 else 0


@pytest.mark.parametrize("compute", [F32, BF16])
@pytest.mark.parametrize("kind", [INT8, INT4])
def test_partials_query_keeps_the_line(kind, compute):
    query = capi.lib().caifx_qlinear_partials_workspace_bytes
    for M, N, K in itertools.product([3, 16, 17, 32], [16, 1024, 8192, 8256, 32768, 40000, 200000, 1 << 20],
                                     [128, 2048, 2176, 4096, 4224, 14336, 65536, 131072, 262144]):
        got, counted = query(M, N, K, compute, compute, kind, 0), _counted(M, N, K, compute, kind)
        if not (compute == F32 and kind == INT4):      # int4 with fp32 compute is the fp32 kernel's alone
            assert got >= counted
            assert (got > LIMIT) == (max(counted, _tiled(M, N, K, compute, kind)) > LIMIT), (M, N, K, got, counted)


def _tiled(M, N, K, compute, kind):
    # what the tiled kernel's shared reduction asks for: up to 8 parts of at least 8 steps of 64 for at most 128 tiles
    tiles = -(-M // 128) * -(-N // 128)
    if tiles > 128 or K % 64:
        return 0
    parts = min(256 // tiles, 8, K // 64 // 8)
    return parts * M * N * 4 if parts >= 2 else 0


def test_degenerate_sizes():
    # refused calls (no rows, no reduction) ask for nothing, a reduction that is no multiple of 64 fits no kernel that shares it
    query = capi.lib().caifx_qlinear_workspace_bytes
    for M, N, K in [(0, 64, 128), (4, 64, 0), (4, 64, 100)]:
        assert query(M, N, K, BF16, BF16, INT8, 0) == 0
