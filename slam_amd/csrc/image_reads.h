// image_reads.h -- reads of several bytes at any place of an 8-bit image that
// stay inside it.  For host and device: a read's bounds are checked on the CPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define IMAGE_HD __host__ __device__ __forceinline__
#else
#define IMAGE_HD inline
#endif

namespace slam {

// The first three bytes of texel (x, y) of a colour image (w x h texels of ch
// = 3 or 4 bytes, rows `pitch` bytes apart) are the low bytes of the 4-byte
// word at `offset`, shifted right by 8 * early bits: the last texel of a
// three-byte image is read one byte early, as no byte need follow it.
struct TexelRead {
    size_t offset;
    int early;
};

IMAGE_HD TexelRead texel_read(int x, int y, int w, int h, int pitch, int ch)
{
    const int early = (x == w - 1 && y == h - 1 && ch == 3) ? 1 : 0;
    return {(size_t)y * pitch + (size_t)x * ch - early, early};
}

// The bytes of T from column x (-2 or more) of row y of an image of n bytes
// (row length w, n at least sizeof(T)); bytes outside the image are 0.
template <class T>
IMAGE_HD T row_bytes(const uint8_t* __restrict__ img, int n, int w, int y, int x)
{
    constexpr int B = sizeof(T);
    const int want = y * w + x, last = n - B;
    const int at = want < 0 ? 0 : (want > last ? last : want);
    T v;
    __builtin_memcpy(&v, img + at, B);
    const int past = want - at < B - 1 ? want - at : B - 1;
    return want < at ? v << (8 * (at - want)) : v >> (8 * past);
}

}  // namespace slam
