"""Pixel order of a window's samples (csrc/pixel_order.h), compiled for the
host: every pixel once, strips of 8 rows column by column, and images of up
to 2^30 pixels in one row without overflow."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    src, so = d / "order.cpp", d / "order.so"
    src.write_text("#define RT_HD inline\n"
                   f'#include "{ROOT}/3d-ray_amd/csrc/pixel_order.h"\n'
                   'extern "C" int order(int q, int W, int npix) { return rt::pixel_of_rank(q, W, npix); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-ftrapv", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    return C.CDLL(str(so)).order


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
