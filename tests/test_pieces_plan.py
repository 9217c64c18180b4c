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
