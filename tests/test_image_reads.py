"""The kernels' reads of several bytes at a time (image_reads.h), compiled for
the CPU: every read lies inside an image that ends with its last texel's last
byte, and gives the bytes that single reads give."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

SOURCE = """
#include "image_reads.h"
#include <string.h>
using namespace slam;
// 0, or 1 + the index of the first texel whose read leaves the image or is wrong
extern "C" long check_texels(const uint8_t* img, long bytes, int w, int h, int pitch, int ch)
{
    for (int y = 0; y < h; ++y)
        for (int x = 0; x < w; ++x) {
            const TexelRead t = texel_read(x, y, w, h, pitch, ch);
            const uint8_t* px = img + (size_t)y * pitch + (size_t)x * ch;
            if (t.offset + 4 > (size_t)bytes) return 1 + (long)y * w + x;
            uint32_t v;
            memcpy(&v, img + t.offset, 4);
            v >>= 8 * t.early;
            for (int k = 0; k < 3; ++k)
                if (((v >> (8 * k)) & 255) != px[k]) return 1 + (long)y * w + x;
        }
    return 0;
}
// The same for groups of G pixels of a row, from two columns before the first.
template <class T, int G>
long check_rows(const uint8_t* img, int w, int h)
{
    for (int y = 0; y < h; ++y)
        for (int x0 = 0; x0 < w; x0 += G) {
            const T v = row_bytes<T>(img, w * h, w, y, x0 - 2);
            for (int k = 0; k < (int)sizeof(T); ++k) {
                const long at = (long)y * w + x0 - 2 + k;
                const int want = at >= 0 && at < (long)w * h ? img[at] : 0;
                if ((int)((v >> (8 * k)) & 255) != want) return 1 + (long)y * w + x0;
            }
        }
    return 0;
}
extern "C" long check_rows_1(const uint8_t* img, int w, int h) { return check_rows<uint32_t, 1>(img, w, h); }
extern "C" long check_rows_4(const uint8_t* img, int w, int h) { return check_rows<uint64_t, 4>(img, w, h); }
"""


@pytest.fixture(scope="module")
def reads(tmp_path_factory):
    d = tmp_path_factory.mktemp("reads")
    (d / "reads.cpp").write_text(SOURCE)
    out = d / "libreads.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                    "-I" + os.path.join(ROOT, "slam_amd", "csrc"), str(d / "reads.cpp"), "-o", str(out)], check=True)
    L = ctypes.CDLL(str(out))
    L.check_texels.restype = L.check_rows_1.restype = L.check_rows_4.restype = ctypes.c_long
    return L


def at_the_end_of_a_page(data):
    """A copy of the bytes that ends where readable memory does."""
    import mmap
    page = mmap.PAGESIZE
    size = (len(data) + page - 1) // page * page
    m = mmap.mmap(-1, size + page)
    base = ctypes.addressof(ctypes.c_char.from_buffer(m))
    libc = ctypes.CDLL(None, use_errno=True)
    assert libc.mprotect(ctypes.c_void_p(base + size), ctypes.c_size_t(page), 0) == 0
    ptr = base + size - len(data)
    ctypes.memmove(ptr, data, len(data))
    return m, ptr


@pytest.mark.parametrize("ch,pad", [(3, 0), (3, 1), (3, 5), (4, 0), (4, 3)])
@pytest.mark.parametrize("w,h", [(16, 16), (17, 16), (65, 32), (131, 97)])
def test_texel_reads_stay_inside(reads, w, h, ch, pad):
    pitch = w * ch + pad
    img = np.random.default_rng(w + ch).integers(0, 256, pitch * (h - 1) + w * ch).astype(np.uint8).tobytes()
    m, ptr = at_the_end_of_a_page(img)
    assert reads.check_texels(ctypes.c_void_p(ptr), ctypes.c_long(len(img)), w, h, pitch, ch) == 0


@pytest.mark.parametrize("w,h", [(4, 4), (5, 4), (6, 5), (7, 4), (16, 16), (53, 40), (131, 97)])
def test_row_reads_stay_inside(reads, w, h):
    img = np.random.default_rng(w).integers(0, 256, w * h).astype(np.uint8).tobytes()
    m, ptr = at_the_end_of_a_page(img)
    assert reads.check_rows_1(ctypes.c_void_p(ptr), w, h) == 0
    assert reads.check_rows_4(ctypes.c_void_p(ptr), w, h) == 0
