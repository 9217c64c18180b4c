"""The C library builds without Python and torch: only the torch_calls target looks for their headers."""
import subprocess

from caif_amd import capi


def test_the_library_alone_asks_for_no_python():
    def commands(*targets):
        return subprocess.run(["make", "-n", "-B", "-C", capi.CSRC, "PYTHON=no-such-python", *targets], check=True, capture_output=True,
                              text=True).stdout
    default = commands()
    assert "libcaifx.so" in default and "torch_calls" not in default and "include/python" not in default
    assert "torch_calls.cpp" in commands("torch_calls")
