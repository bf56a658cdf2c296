// pyramid.hpp -- one HALF Gaussian pyramid step (ScaleGaussianHalf 5x5) as a device routine, shared by
// the per-node kernel and the frame-batched graph.
//
// HafCpu_ScaleGaussianHalf_U8_U8_5x5 (ago_haf_cpu_pyramid.cpp:94-305), wrapper ago_kernel_api.cpp:15420-15436:
// out(x, y) = (sum_j k_j H(2y+oy-2+j)) >> 8, H(r) = sum_i k_i p(2x+ox-2+i, r), k = [1 4 6 4 1],
// oy = (srcH even), ox = (srcW even), rows 1..dh-2, linear-address taps with the zero guard.
#pragma once
#include "mvx_common.hpp"
#include <algorithm>

namespace mvx {

// A wave computes one output row of 62 chunks of 8 columns: lane l holds the 16 source bytes of chunk
// firstChunk + l - 1 of the five source rows (lanes 0 and 63 only feed their neighbours).  Vertical sums
// first, on byte pairs split into even and odd columns (two 16-bit values a register: at most 16 * 255),
// then the horizontal taps, whose neighbours past the chunk come from the next lanes by three DPP shifts; a
// result is at most 256 * 255, so nothing wraps.  Short waves on purpose: the levels of a pyramid are small
// and follow each other, so what counts is the time of one wave.  With 8 columns x 4 rows a thread, bytes
// unpacked one by one and 11 rows loaded in turn, a level took 7 to 10 us down to the smallest sizes; five
// independent 16-byte loads and about 140 instructions make it 3 us for the small ones (3840x2160 to 1920x1080: 10.4 -> 6.2 us).
constexpr int PYR_CHUNKS = 62;

MVX_DEV u16x2 pyr_from_prev(u16x2 v) { return pair_of((uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits_of(v), 0x138, 0xf, 0xf, true)); }
MVX_DEV u16x2 pyr_from_next(u16x2 v) { return pair_of((uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits_of(v), 0x130, 0xf, 0xf, true)); }
// 1 4 6 4 1
MVX_DEV u16x2 pyr_taps(u16x2 a, u16x2 b, u16x2 c, u16x2 d, u16x2 e)
{
    return (a + e) + (b + d) * (unsigned short)4 + c * (unsigned short)6;
}

// output row y (1..dh-2, the same in the whole wave), chunks firstChunk .. firstChunk + PYR_CHUNKS - 1; every
// lane of the wave calls it
MVX_DEV void half_row(uint32_t dw, uint8_t *dst, uint32_t dstStride, uint32_t sw, uint32_t sh, const uint8_t *src, uint32_t srcStride,
                      uint32_t firstChunk, int y)
{
    const int lane = (int)threadIdx.x & 63;
    const long chunk = (long)firstChunk + lane - 1;
    const long n = (long)sh * srcStride;
    const int oy = (sh & 1) ? 0 : 1;
    const long row0 = (long)(2 * y + oy - 2) * srcStride;
    uint4 p[5];
#pragma unroll
    for (int j = 0; j < 5; j++) {
        const long off = row0 + (long)j * srcStride + 16 * chunk;   // linear addresses, zeros outside the plane
        p[j] = (off < 0 || off >= n) ? make_uint4(0, 0, 0, 0) : *reinterpret_cast<const uint4 *>(src + off);
    }
    u16x2 E[6], O[6];   // vertical sums of columns 4d, 4d+2 and 4d+1, 4d+3 of dword d at [d + 1]
#pragma unroll
    for (int d = 0; d < 4; d++) {
        u16x2 e[5], o[5];
#pragma unroll
        for (int j = 0; j < 5; j++) {
            const uint32_t v = d == 0 ? p[j].x : d == 1 ? p[j].y : d == 2 ? p[j].z : p[j].w;
            e[j] = even_bytes(v);
            o[j] = odd_bytes(v);
        }
        E[d + 1] = pyr_taps(e[0], e[1], e[2], e[3], e[4]);
        O[d + 1] = pyr_taps(o[0], o[1], o[2], o[3], o[4]);
    }
    u16x2 r[4];
    if (sw & 1) {   // centres 2x
        E[0] = pyr_from_prev(E[4]); O[0] = pyr_from_prev(O[4]);
        E[5] = pyr_from_next(E[1]);
#pragma unroll
        for (int d = 1; d <= 4; d++)
            r[d - 1] = pyr_taps(pair_shift(E[d - 1], E[d]), pair_shift(O[d - 1], O[d]), E[d], O[d], pair_shift(E[d], E[d + 1]));
    } else {        // centres 2x + 1
        O[0] = pyr_from_prev(O[4]);
        E[5] = pyr_from_next(E[1]); O[5] = pyr_from_next(O[1]);
#pragma unroll
        for (int d = 1; d <= 4; d++)
            r[d - 1] = pyr_taps(pair_shift(O[d - 1], O[d]), E[d], O[d], pair_shift(E[d], E[d + 1]), pair_shift(O[d], O[d + 1]));
    }
    const uint2 v = make_uint2(__builtin_amdgcn_perm(bits_of(r[1]), bits_of(r[0]), 0x07050301u),
                               __builtin_amdgcn_perm(bits_of(r[3]), bits_of(r[2]), 0x07050301u));
    const long x0 = 8 * chunk;
    if (lane == 0 || lane == 63 || x0 >= (long)dw) return;
    uint8_t *out = dst + (long)y * dstStride + x0;
    if (x0 + 8 <= (long)dw) {
        *reinterpret_cast<uint2 *>(out) = v;
    } else {
        for (int i = 0; x0 + i < (long)dw; i++) out[i] = (uint8_t)((i < 4 ? v.x : v.y) >> (8 * (i & 3)));
    }
}

// the grid of a level: 4 rows a workgroup (64 x 4 threads); the rows of a plane too tall for one grid wrap round
inline dim3 half_grid(uint32_t dw, uint32_t dh, uint32_t planes)
{
    return dim3(((dw + 7) / 8 + PYR_CHUNKS - 1) / PYR_CHUNKS, std::min((dh - 2 + 3) / 4, 65535u), planes);
}

}  // namespace mvx
