"""Tiles and shared reductions of the products of bf16 pieces (fp32 compute), which are chosen on the host: what the launch and the
workspace can hold, for calls over the whole accepted range."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NO_LIMIT = 2 ** 63
STATIC = 8 << 20


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "pieces_plan")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "caif_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pieces_plan.cpp"), "-o", exe], check=True)

    def ask(calls):
        text = "".join("%d %d %d %d %d\n" % c for c in calls)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
        assert len(out) == len(calls)
        return [tuple(int(v) for v in line.split()) for line in out]
    return ask


CALLS = list(itertools.product([1, 2, 16, 33, 64, 65, 100, 128, 129, 200, 999, 2048, 4096, 65536, 2097120, 2097121, 2 ** 22 - 1, 2 ** 22],
                               [16, 64, 512, 1408, 4096, 14336], [64, 128, 192, 256, 512, 640, 2048, 4096, 14336], [0, 1],
                               [0, 1 << 16, 1 << 20, NO_LIMIT]))


def test_every_plan_fits_the_launch_and_the_room(plans):
    for (M, C, R, int4, room), (bm, parts, per, size) in zip(CALLS, plans(CALLS)):
        assert bm in (32, 64, 128)
        assert -(-M // bm) <= 65535, (M, C, R, int4, bm)          # gridDim.y
        assert 1 <= parts <= 65535 and (parts - 1) * per < R // 64 <= parts * per
        assert size == (parts * M * C * 4 if parts > 1 else 0) and size <= min(room, STATIC)


# One or two steps in more than one round of the chip, where tiles of 32 rows cut the weight four times as often: int8, us with 32 / 64 /
# 128 rows 215 / 174 / 165, 118 / 94 / 97, 60 / 53 / 51, 54 / 47 / 46, 133 / 117 / 115 in the order
# below (int4 161 / 142 / 152 to 44 / 40 / 43; with one step 102 / 97 / 104, left out).
@pytest.mark.parametrize("int4", [0, 1])
def test_short_reductions_of_many_rows_take_tall_tiles(plans, int4):
    calls = [(M, C, R, int4, room) for M, C, R in [(4096, 14336, 128), (4096, 8192, 128), (4096, 4096, 128), (1024, 14336, 128), (4096, 14336, 64)][:4 if int4 else 5]
             for room in (0, NO_LIMIT)]
    assert all(bm > 32 for bm, _, _, _ in plans(calls))
