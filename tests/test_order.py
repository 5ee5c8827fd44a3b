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
                      'extern "C" int split(int v, int tiles, int slices, int tiles_first, int* slice) {\n'
                      '  const lt_split_place at = tiles_first ? lt_split_by_tile(v, tiles, slices) : lt_split_by_slice(v, tiles, slices);\n'
                      '  *slice = at.slice;\n  return at.tile;\n}\n'
                      'extern "C" int tiles_first(int64_t m, int64_t n, int64_t k) { return lt_split_tiles_first(m, n, k); }\n'
                      'extern "C" int can_stagger(int nseg, int64_t k) { return lt_can_stagger(nseg, k); }\n')
    subprocess.run([compiler, "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(library)], check=True)
    lib = ctypes.CDLL(str(library))
    lib.tiles_first.argtypes = [ctypes.c_int64] * 3
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


@pytest.mark.parametrize("tiles,slices", [(1, 2), (3, 5), (8, 16), (32, 16), (36, 7), (84, 3), (91, 2), (200, 2)])
@pytest.mark.parametrize("tiles_first", [False, True])
def test_tiles_and_slices_of_a_split_product(order, tiles, slices, tiles_first):
    """every tile of every slice once; an XCD's own follow each other, tile by tile or slice by slice"""
    slice_ = ctypes.c_int()
    places = []
    for v in range(tiles * slices):
        tile = order.split(v, tiles, slices, tiles_first, ctypes.byref(slice_))
        places.append(tile * slices + slice_.value if tiles_first else slice_.value * tiles + tile)
    assert sorted(places) == list(range(tiles * slices))
    for xcd in range(8):
        own = places[xcd::8]
        assert own == list(range(own[0], own[0] + len(own))) if own else tiles * slices <= xcd


def test_which_split_products_go_tile_by_tile(order):
    """a large operand streamed against a thin one: yes; one of up to 64 MiB, or both used by several tiles: no"""
    assert order.tiles_first(4096, 128, 16384) and order.tiles_first(4096, 8, 16384) and order.tiles_first(129, 4096, 16384)
    assert not order.tiles_first(4096, 128, 8192) and not order.tiles_first(1000, 64, 16384) and not order.tiles_first(128, 4096, 8192)
    assert not order.tiles_first(4096, 136, 16384) and not order.tiles_first(257, 4096, 32768)
