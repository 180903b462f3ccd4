"""Pixel order of a window's samples and block order of a launch
(csrc/pixel_order.h), compiled for the host: every pixel once, strips of 8
rows column by column, images of up to 2^30 pixels in one row without
overflow; every block once, and the XCDs' shares of an image's columns."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    src, so = d / "order.cpp", d / "order.so"
    src.write_text("#define RT_HD inline\n"
                   f'#include "{ROOT}/3d-ray_amd/csrc/pixel_order.h"\n'
                   'extern "C" int order(int q, int W, int npix) { return rt::pixel_of_rank(q, W, npix); }\n'
                   'extern "C" uint32_t remap(uint32_t b, uint32_t nb, uint32_t run) '
                   '{ return rt::xcd_remap(b, nb, run); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-ftrapv", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    return C.CDLL(str(so))


@pytest.fixture(scope="module")
def order(lib):
    return lib.order


@pytest.fixture(scope="module")
def remap(lib):
    lib.remap.argtypes = [C.c_uint32] * 3
    lib.remap.restype = C.c_uint32
    return lib.remap


@pytest.mark.parametrize("W,H", [(1, 1), (5, 3), (1, 40), (64, 8), (13, 17), (9, 7)])
def test_strips(order, W, H):
    got = [order(q, W, W * H) for q in range(W * H)]
    want = [y * W + x for y0 in range(0, H, 8) for x in range(W) for y in range(y0, min(y0 + 8, H))]
    assert got == want


@pytest.mark.parametrize("W,H", [(1 << 30, 1), (1 << 29, 2), (1 << 28, 4), ((1 << 28) + 7, 3), (1 << 27, 8), (107374182, 10)])
def test_widest_images(order, W, H):
    n = W * H
    rng = np.random.default_rng(3)
    for q in [0, 1, n // 2, n - 1] + [int(v) for v in rng.integers(0, n, 200)]:
        y0 = q // (8 * W) * 8
        h = min(8, H - y0)
        x, y = divmod(q - y0 * W, h)
        assert order(q, W, n) == (y0 + y) * W + x, (q, W, H)


@pytest.mark.parametrize("nb,longest", [(1, 1), (7, 4), (64, 1), (1000, 4), (3293, 32), (4096, 10), (5000, 2), (20000, 32)])
def test_block_order_is_a_permutation(remap, nb, longest):
    assert sorted(remap(b, nb, longest) for b in range(nb)) == list(range(nb))


@pytest.mark.parametrize("strip", list(range(2, 41)))
def test_xcds_share_the_columns(remap, strip):
    # an image of strips of `strip` runs whose left half is sky: no XCD has
    # much more of the other half than the rest (in a fixed order one could
    # have all of it); 64 rounds of eight runs
    run, rounds = 4, 64
    nb = 8 * run * rounds
    busy = np.zeros(8)
    for b in range(nb):
        r = remap(b, nb, run) // run
        busy[b % 8] += (r % strip) >= strip / 2
    assert busy.max() < 1.2 * busy.mean(), busy / busy.mean()
