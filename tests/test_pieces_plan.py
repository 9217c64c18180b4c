"""Tiles and shared reductions of the products of bf16 pieces (fp32 compute), which are chosen on the host: what the launch and the
workspace can hold, for calls over the whole accepted range."""
import itertools

import pytest

NO_LIMIT = 2 ** 63
STATIC = 8 << 20


CALLS = list(itertools.product([1, 2, 16, 33, 64, 65, 100, 128, 129, 200, 999, 2048, 4096, 65536, 2097120, 2097121, 2 ** 22 - 1, 2 ** 22],
                               [16, 64, 512, 1408, 4096, 14336], [64, 128, 192, 256, 512, 640, 2048, 4096, 14336], [0, 1],
                               [0, 1 << 16, 1 << 20, NO_LIMIT]))


def test_every_plan_fits_the_launch_and_the_room(pieces_plans):
    for (M, C, R, int4, room), (bm, parts, per, size, _) in zip(CALLS, pieces_plans(CALLS)):
        assert bm in (32, 64, 128)
        assert -(-M // bm) <= 65535, (M, C, R, int4, bm)          # gridDim.y
        assert 1 <= parts <= 65535 and (parts - 1) * per < R // 64 <= parts * per
        assert size == (parts * M * C * 4 if parts > 1 else 0) and size <= min(room, STATIC)


# One or two steps in more than one round of the chip, where tiles of 32 rows cut the weight four times as often: int8, us with 32 / 64 /
# 128 rows 215 / 174 / 165, 118 / 94 / 97, 60 / 53 / 51, 54 / 47 / 46, 133 / 117 / 115 in the order
# below (int4 161 / 142 / 152 to 44 / 40 / 43; with one step 102 / 97 / 104, left out).
@pytest.mark.parametrize("int4", [0, 1])
def test_short_reductions_of_many_rows_take_tall_tiles(pieces_plans, int4):
    calls = [(M, C, R, int4, room) for M, C, R in [(4096, 14336, 128), (4096, 8192, 128), (4096, 4096, 128), (1024, 14336, 128), (4096, 14336, 64)][:4 if int4 else 5]
             for room in (0, NO_LIMIT)]
    assert all(bm > 32 for bm, *_ in pieces_plans(calls))


# Up to 128 rows without room to share the reduction: the pieces' one chain of steps takes 76 (int4) and 92 us (int8) at 4096, 40 and 49 at
# 2048, whatever the rows and columns of a chip that is not full; the fp32 instruction's split tile takes 43 and 45, 23 and 24.
@pytest.mark.parametrize("int4", [0, 1])
def test_without_room_the_faster_kernel_takes_the_call(pieces_plans, int4):
    sizes = list(itertools.product([33, 64, 100, 128], [64, 512, 1024, 2048], [1024, 2048, 4096]))
    assert all(split for *_, split in pieces_plans([(M, C, R, int4, 0) for M, C, R in sizes]))
    assert not any(split for *_, split in pieces_plans([(M, C, R, int4, NO_LIMIT) for M, C, R in sizes]))
    # not where its larger tiles would have to, nor where the chip is full
    assert not any(split for *_, split in pieces_plans([(M, C, R, int4, 0) for M, C, R in [(129, 512, 4096), (200, 1024, 2048), (64, 512, 2112), (128, 14336, 4096)]]))


# with room too where the reduction is short: int8, us on the pieces (their best plan) and on the split tile 9.1 / 6.8, 9.8 / 6.9, 7.1 / 4.9
def test_short_reductions_of_few_rows(pieces_plans):
    assert all(split for *_, split in pieces_plans([(M, C, R, 0, NO_LIMIT) for M, C, R in [(100, 1024, 256), (100, 2048, 256), (128, 512, 128)]]))
    assert not any(split for *_, split in pieces_plans([(M, C, R, 0, NO_LIMIT) for M, C, R in [(200, 1024, 256), (100, 1024, 192)]]))
