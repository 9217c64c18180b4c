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


def _plans(tmp_path_factory, name, number=int):
    """Asks tests/cpp/<name>.cpp, a host program around the library's own header, for the plan of each call: numbers in, numbers out."""
    exe = str(tmp_path_factory.mktemp("plan") / name)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "caif_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp"), "-o", exe], check=True)

    def ask(calls):
        text = "".join(" ".join("%d" % v for v in c) + "\n" for c in calls)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
        assert len(out) == len(calls)
        return [tuple(number(v) for v in line.split()) for line in out]
    return ask


@pytest.fixture(scope="session")
def pieces_plans(tmp_path_factory):
    """What the host chooses for fp32-compute calls (M, columns, reduction, int4, room): rows of a tile, workgroups per reduction, their
    steps, bytes of their sums, and whether the fp32 instruction's split tile takes the call instead."""
    return _plans(tmp_path_factory, "pieces_plan")


@pytest.fixture(scope="session")
def tall_plans(tmp_path_factory):
    """Height of the tall kernel's row tiles for grouped int8 calls (rows, experts, columns, reduction), and the estimate in us."""
    return _plans(tmp_path_factory, "tall_plan", float)


@pytest.fixture(scope="session")
def few_plans(tmp_path_factory):
    """How the few-row forward kernel cuts calls (rows, columns, reduction, kind): row tiles, their 16-row blocks, workgroups per reduction
    and the units of each; zeros where another kernel takes the call."""
    return _plans(tmp_path_factory, "few_plan")
