"""The pixel order of a top-level camera launch, compiled for the host: every pixel once, and nothing out of range."""

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "bajo_amd" / "csrc"
SOURCE = """
#include "pixel_order.h"
extern "C" void pixels(const uint64_t* r, uint64_t count, uint64_t R, uint32_t w, uint32_t h, uint64_t* out) {
  for (uint64_t i = 0; i < count; ++i) out[i] = bj::camera_pixel(r[i], R, w, h);
}
"""


@pytest.fixture(scope="module")
def pixels(tmp_path_factory):
    d = tmp_path_factory.mktemp("pixel_order")
    (d / "p.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(d / "p.so"), str(d / "p.cpp")], check=True)
    fn = ctypes.CDLL(str(d / "p.so")).pixels
    u64 = np.ctypeslib.ndpointer(np.uint64, flags="C_CONTIGUOUS")
    fn.argtypes = [u64, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint32, u64]

    def run(r, R, w, h):
        r = np.ascontiguousarray(r, np.uint64)
        out = np.empty_like(r)
        fn(r, r.size, R, w, h, out)
        return out

    return run


@pytest.mark.parametrize("w,h,views,cut", [(1, 1, 3, 0), (8, 8, 1, 0), (9, 7, 2, 5), (640, 360, 1, 0), (37, 21, 2, 0),
                                           (70, 30, 2, 1000), (1, 200, 1, 0), (200, 1, 2, 0), (5000, 9, 1, 0)])
def test_every_pixel_once(pixels, w, h, views, cut):
    R = w * h * views - cut
    out = pixels(np.arange(R), R, w, h)
    np.testing.assert_array_equal(np.sort(out), np.arange(R, dtype=np.uint64))


@pytest.mark.parametrize("w,h", [((1 << 31) - 1, 1), (1 << 30, 1), ((1 << 29) + 3, 3), (1 << 29, 2), (1 << 28, 7),
                                 ((1 << 28) - 1, 8), ((1 << 27) + 1, 15), (3, (1 << 29) + 1), (1, (1 << 31) - 1)])
def test_very_wide_and_very_high_views(pixels, w, h):
    """Widths from 2^29 made 8 w wrap to 0 in 32 bits: sampled indices stay in the view and stay distinct, and the
    tile that holds an index is the one it should be (counted in Python's integers)."""
    R = w * h
    rng = np.random.default_rng(w % 1000 + h)
    r = np.unique(np.concatenate([rng.integers(0, R, 20_000), [0, 1, R // 2, R - 2, R - 1]]).astype(np.uint64))
    out = pixels(r, R, w, h)
    assert out.max() < R and np.unique(out).size == out.size
    for i in range(0, r.size, 997):
        k = int(r[i])
        band, k = divmod(k, 8 * w)
        rows = min(8, h - 8 * band)
        tile, k = divmod(k, 8 * rows)
        cols = min(8, w - 8 * tile)
        y, x = divmod(k, cols)
        assert int(out[i]) == (8 * band + y) * w + 8 * tile + x
