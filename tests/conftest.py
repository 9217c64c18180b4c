import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def orc():
    """The CPU oracle (test infrastructure; builds with gcc in seconds)."""
    from oracle import oracle
    oracle.build()
    return oracle


@pytest.fixture(scope="session")
def pieces_plans(tmp_path_factory):
    """What the host chooses for fp32-compute calls (M, columns, reduction, int4, room): rows of a tile, workgroups per reduction, their
    steps, bytes of their sums, and whether the fp32 instruction's split tile takes the call instead."""
    exe = str(tmp_path_factory.mktemp("plan") / "pieces_plan")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "caif_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pieces_plan.cpp"), "-o", exe], check=True)

    def ask(calls):
        text = "".join("%d %d %d %d %d\n" % c for c in calls)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
        assert len(out) == len(calls)
        return [tuple(int(v) for v in line.split()) for line in out]
    return ask
