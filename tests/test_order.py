"""Which tile and slice the workgroups of a launch take (csrc/lt_order.h): on the host, in plain C++.  Workgroup v runs on XCD v % 8."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lean_transformer_amd", "csrc")


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no C++ compiler")
    folder = tmp_path_factory.mktemp("order")
    source, library = folder / "order.cpp", folder / "order.so"
    source.write_text('#include "lt_order.h"\n'
                      'extern "C" int tile(int v, int m, int n, int staggered) { return lt_tile_order(v, m, n, staggered); }\n'
                      'extern "C" int can_stagger(int nseg, int64_t k) { return lt_can_stagger(nseg, k); }\n')
    subprocess.run([compiler, "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(library)], check=True)
    lib = ctypes.CDLL(str(library))
    lib.can_stagger.argtypes = [ctypes.c_int, ctypes.c_int64]
    return lib


@pytest.mark.parametrize("m,n", [(1, 1), (1, 8), (3, 5), (7, 45), (7, 12), (10, 47), (11, 47), (14, 25), (16, 64), (31, 36)])
@pytest.mark.parametrize("staggered", [False, True])
def test_tiles_of_an_unsplit_product(order, m, n, staggered):
    """every tile once; few rows under the stagger: neighbours on neighbouring XCDs; else an XCD's tiles follow each other"""
    tiles = [order.tile(v, m, n, staggered) for v in range(m * n)]
    assert sorted(tiles) == list(range(m * n))
    if staggered and m <= 10 and m * n % 8:
        assert tiles == list(range(m * n))
    else:
        for xcd in range(8):
            own = tiles[xcd::8]
            assert own == list(range(own[0], own[0] + len(own))) if own else m * n <= xcd


def test_where_the_walk_over_k_can_be_staggered(order):
    assert order.can_stagger(1, 64) and order.can_stagger(1, 11520)
    assert not order.can_stagger(1, 11616) and not order.can_stagger(1, 8) and not order.can_stagger(2, 64)
