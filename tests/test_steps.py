"""Which k-steps of a one- or two-segment reduction the register-staged kernel may load without a test for their end
(csrc/lt_steps.h), against a walk over the steps one by one: on the host, in plain C++."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lean_transformer_amd", "csrc")


@pytest.fixture(scope="module")
def leading_whole_steps(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no C++ compiler")
    folder = tmp_path_factory.mktemp("steps")
    source, library = folder / "steps.cpp", folder / "steps.so"
    source.write_text('#include "lt_steps.h"\n'
                      'extern "C" int steps(int64_t k0, int64_t k1, int step) { return lt_leading_whole_steps(k0, k1, step); }\n')
    subprocess.run([compiler, "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(library)], check=True)
    fn = ctypes.CDLL(str(library)).steps
    fn.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return fn


@pytest.mark.parametrize("k0", [8, 56, 64, 72, 128, 16392, 16384])
@pytest.mark.parametrize("k1", [0, 8, 64, 72, 128])
def test_leading_whole_steps(leading_whole_steps, k0, k1):
    lengths = [min(64, k - start) for k in (k0, k1) for start in range(0, k, 64)]
    whole = next((i for i, n in enumerate(lengths) if n < 64), len(lengths))
    assert leading_whole_steps(k0, k1, 64) == whole
