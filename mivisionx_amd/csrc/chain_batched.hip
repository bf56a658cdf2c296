// chain_batched.hip -- Gaussian3x3 -> Sobel3x3 (gx, gy) -> Magnitude + Phase, plus ScaleImage to half
// size, for a batch of U8 images of uneven sizes in ONE persistent launch.
//
// Per image the launch computes exactly what five reference nodes compute one after another
// (HafCpu_Gaussian_U8_U8_3x3 ago_haf_cpu_filter.cpp:1681-1861 into a virtual image,
// HafCpu_Sobel_S16S16_U8_3x3_GXY :2237, HafCpu_Magnitude_S16_S16S16 ago_haf_cpu_arithmetic.cpp:4989,
// HafCpu_Phase_U8_S16S16 :9592, HafCpu_ScaleImage_U8_U8_Bilinear ago_haf_cpu_geometric.cpp:1977 on
// the input), but the blurred image never leaves registers.
//
// Lanes and tiles.  A lane owns 8 columns and streams down its rows, everything in registers: the input
// rows' vertical sums, the blurred rows and the gradients are pairs of 16-bit columns, and the one or two
// columns it needs on either side come with its own loads (16 bytes from 4 left of its columns), so no
// lane waits for another and there is no LDS and no barrier.  Every byte is the one at LINEAR index
// r*stride + c of the plane (0 outside [0, h*stride)): the reference reads 3x3 neighbours by linear address,
// so the left neighbour of column 0 is the previous row's last byte and the right neighbour of column w-1
// is padding or the next row's first byte.  A blurred pixel is nonzero only on rows 1..h-2 and columns < w,
// because the Gaussian node writes nothing else and the plane starts zeroed.  Rows 0 and h-1 of gx/gy are
// not written (the Sobel node leaves them); Magnitude and Phase of those rows are computed from zero
// gradients, which is what the nodes compute from the zeroed rows.  The half-size image comes from the same
// input rows.
// An output tile is TW pixels of at most TH rows of one image, TW / 8 lanes; a wave takes tiles that follow each
// other, and an image's tiles are counted up to whole waves, so a wave's lanes share one image.  Tiles are
// lower where all together would leave SIMDs idle, and where an image has too few to fill its waves' lanes
// (the two rows above and below a lane's rows are read and blurred again).
//
// Bound by memory and VALU issue alike: 8.25 bytes and 55 lane operations a pixel.  48 uneven images of
// 118 Mpixel: 349 us with tiles in LDS (73 operations a pixel, a third of them blurring halos and unpacking
// bytes twice), 283 us now.
//
// Schedule.  The waves' tiles of all images form one sequence (image after image, row-major inside an
// image).  The grid is persistent: it is a multiple of 8 workgroups, workgroup b runs on XCD b%8
// (MI355X dispatches workgroups round-robin over its 8 XCDs), the sequence is cut into 8 equal
// contiguous ranges, one per XCD, and the waves of an XCD stride through its range, so tiles
// that share halo rows are processed at the same time on the same L2.  No atomics: the schedule is
// static, so a captured hipGraph replays without any reset.
#include "arith.hpp"
#include <algorithm>
#include <cstring>
#include <vector>

namespace mvx {

struct ChainRow {  // device plan: one 128-byte row per image
    const uint8_t *src;
    int16_t *gx, *gy, *mag;
    uint8_t *phase, *half;
    uint32_t w, h;
    uint32_t srcStride, gxStride, gyStride, magStride, phaseStride, halfStride;
    uint32_t tilesX, tileBegin;  // tiles per row; index of the image's first tile in the sequence
    uint32_t rows;               // of a tile: even, a divisor of TH
    uint32_t pad[9];
};
static_assert(sizeof(ChainRow) == 128, "plan row is 128 bytes");

// image of tile t: the last plan row with tileBegin <= t (uniform across the wave)
MVX_DEV uint32_t find_image(const ChainRow *__restrict__ plan, uint32_t count, uint32_t t)
{
    uint32_t lo = 0, hi = count - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (plan[mid].tileBegin <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

constexpr int CHAIN_THREADS = 256;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_dword __attribute__((aligned(4)));   // at a 4-byte aligned address

// the plane pointers come out of the plan: as global memory (flat accesses take the LDS counter along)
template <class T> MVX_DEV gptr_t<T> at(const void *base, long offset) { return (gptr_t<T>)(gmem((const uint8_t *)base) + offset); }

// one input row of a lane: dwords c-4, c, c+4, c+8 as column pairs
struct InRow {
    u16x2 E[4], O[4];
};
// one blurred row: columns c-1 (Ol.hi), c..c+7, c+8 (Er.lo)
struct BlurRow {
    u16x2 Ol, E[2], O[2], Er;
};
// the raw input bytes c..c+7 of a row, for the half-size image
struct RawRow {
    uint32_t w[2];
};

// One lane's rows of one image (its tile column x, rows y0 .. y0+rows-1 below h).
struct ChainLane {
    const ChainRow &d;
    int w, h, stride, n, x;
    bool merged, edge;                // edge: some blurred byte it sees may be one the Gaussian node does not write
    uint32_t colE[2], colO[2];        // columns below w
    bool wrapL, wrapR, rightOk;       // column c-1 / c+8 lies in the row above / below; column c+8 is below w
    u16x2 two;                        // {2, 2} the compiler does not see through: multiply-adds instead of shifts and adds

    MVX_DEV u32x4 load(int r) const
    {
        const uint32_t off = (uint32_t)r * (uint32_t)stride + (uint32_t)x - 4u;   // outside the plane: past n, or wrapped far past it
        u32x4 v;
        if (off <= (uint32_t)(n - 16)) {
            v = *at<const u32x4_dword>(d.src, off);
        } else {
            v = u32x4{0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (off + 4u * k <= (uint32_t)(n - 4)) v[k] = *at<const uint32_t>(d.src, off + 4u * k);
        }
        return v;
    }

    MVX_DEV uint32_t row_mask(int r) const { return (uint32_t)(r - 1) < (uint32_t)(h - 2) ? ~0u : 0u; }

    // blurred row r from input rows r-1, r, r+1: (h(r-1) + 2 h(r) + h(r+1)) >> 4 with h = p(c-1) + 2 p(c) + p(c+1),
    // as the Gaussian node computes it (vertical sums first: integers)
    MVX_DEV BlurRow blur(int r, const InRow &a, const InRow &b, const InRow &c) const
    {
        InRow v;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v.E[k] = a.E[k] + b.E[k] * two + c.E[k];
            v.O[k] = a.O[k] + b.O[k] * two + c.O[k];
        }
        const auto even = [&](int k) { return (pair_shift(v.O[k - 1], v.O[k]) + v.O[k] + v.E[k] * two) >> (unsigned short)4; };
        const auto odd = [&](int k) { return (v.E[k] + pair_shift(v.E[k], v.E[k + 1]) + v.O[k] * two) >> (unsigned short)4; };
        BlurRow o{odd(0), {even(1), even(2)}, {odd(1), odd(2)}, even(3)};
        if (edge) {
            const uint32_t m = row_mask(r);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                o.E[k] = pair_of(bits_of(o.E[k]) & colE[k] & m);
                o.O[k] = pair_of(bits_of(o.O[k]) & colO[k] & m);
            }
            o.Ol = pair_of(bits_of(o.Ol) & (x > 0 ? m : wrapL ? row_mask(r - 1) : 0u));
            o.Er = pair_of(bits_of(o.Er) & (rightOk ? m : wrapR ? row_mask(r + 1) : 0u));
        }
        return o;
    }

    MVX_DEV void put_magphase(int y, bool full, u32x4 m, u32x2 p) const
    {
        const long pm = (long)y * d.magStride + 2 * x, pp = (long)y * d.phaseStride + x;
        if (full) {
            *at<u32x4>(d.mag, pm) = m;
            *at<u32x2>(d.phase, pp) = p;
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; j++)   // widths are even
            if (x + 2 * j < w) {
                *at<uint32_t>(d.mag, pm + 4 * j) = m[j];
                *at<uint16_t>(d.phase, pp + 2 * j) = (uint16_t)(p[j >> 1] >> (16 * (j & 1)));
            }
    }

    // Sobel, Magnitude, Phase of row y from blurred rows y-1, y, y+1.  With virtual gradients (gx == gy == NULL)
    // the image takes the merged SobelMagnitudePhase kernel instead: no gradient stores, rows 1..h-2 only,
    // and magnitude columns from w & ~15 on truncate (ago_haf_cpu_filter.cpp:3972-4202).
    MVX_DEV void gradients(int y, const BlurRow &a, const BlurRow &b, const BlurRow &c) const
    {
        const bool full = x + 8 <= w;
        if (row_mask(y) == 0) {   // the Sobel node skips the row; the other nodes see zero gradients
            if (merged) return;
            put_magphase(y, full, u32x4{0, 0, 0, 0}, u32x2{0, 0});
            return;
        }
        uint32_t gxw[4], gyw[4];   // columns of gx and gy in order (16-bit, in [-1020, 1020])
        {
            const auto sum = [this](u16x2 p, u16x2 q, u16x2 r) { return p + q * two + r; };
            const BlurRow s{sum(a.Ol, b.Ol, c.Ol), {sum(a.E[0], b.E[0], c.E[0]), sum(a.E[1], b.E[1], c.E[1])},
                            {sum(a.O[0], b.O[0], c.O[0]), sum(a.O[1], b.O[1], c.O[1])}, sum(a.Er, b.Er, c.Er)};
            const BlurRow f{c.Ol - a.Ol, {c.E[0] - a.E[0], c.E[1] - a.E[1]}, {c.O[0] - a.O[0], c.O[1] - a.O[1]}, c.Er - a.Er};
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint32_t xe = bits_of(s.O[k] - pair_shift(k ? s.O[0] : s.Ol, s.O[k])), xo = bits_of(pair_shift(s.E[k], k ? s.Er : s.E[1]) - s.E[k]);
                const uint32_t ye = bits_of(sum(pair_shift(k ? f.O[0] : f.Ol, f.O[k]), f.E[k], f.O[k]));
                const uint32_t yo = bits_of(sum(f.E[k], f.O[k], pair_shift(f.E[k], k ? f.Er : f.E[1])));
                gxw[2 * k] = __builtin_amdgcn_perm(xo, xe, 0x05040100u);       // columns 4k, 4k+1
                gxw[2 * k + 1] = __builtin_amdgcn_perm(xo, xe, 0x07060302u);   // columns 4k+2, 4k+3
                gyw[2 * k] = __builtin_amdgcn_perm(yo, ye, 0x05040100u);
                gyw[2 * k + 1] = __builtin_amdgcn_perm(yo, ye, 0x07060302u);
            }
            if (!merged) {
                const long px = (long)y * d.gxStride + 2 * x, py = (long)y * d.gyStride + 2 * x;
                if (full) {
                    *at<u32x4>(d.gx, px) = u32x4{gxw[0], gxw[1], gxw[2], gxw[3]};
                    *at<u32x4>(d.gy, py) = u32x4{gyw[0], gyw[1], gyw[2], gyw[3]};
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (x + 2 * j < w) {
                            *at<uint32_t>(d.gx, px + 4 * j) = gxw[j];
                            *at<uint32_t>(d.gy, py + 4 * j) = gyw[j];
                        }
                }
            }
        }
        // the chain's gradients need no distinction of Magnitude's body and tail columns, only the merged
        // kernel's tail truncates
        uint32_t mw[4], pw[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            uint32_t ph[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t gx = gxw[2 * q + (j >> 1)], gy = gyw[2 * q + (j >> 1)];
                const float fx = (float)((j & 1) ? (int32_t)gx >> 16 : (int32_t)(int16_t)gx), fy = (float)((j & 1) ? (int32_t)gy >> 16 : (int32_t)(int16_t)gy);
                const uint32_t m = mag_sobel(fx, fy);
                if (j & 1) mw[2 * q + (j >> 1)] = __builtin_amdgcn_perm(m, mw[2 * q + (j >> 1)], 0x05040100u);
                else mw[2 * q + (j >> 1)] = m;
                ph[j] = phase_sobel(fx, fy);
            }
            pw[q] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(ph[3], ph[2], 0x0c0c0400u), __builtin_amdgcn_perm(ph[1], ph[0], 0x0c0c0400u), 0x05040100u);
        }
        const int body = w & ~15;
        if (merged && x + 8 > body)
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (x + j >= body) {
                    const uint32_t gx = gxw[j >> 1], gy = gyw[j >> 1];
                    const uint32_t m = mag_sobel_trunc((float)((j & 1) ? (int32_t)gx >> 16 : (int32_t)(int16_t)gx),
                                                       (float)((j & 1) ? (int32_t)gy >> 16 : (int32_t)(int16_t)gy));
                    mw[j >> 1] = (j & 1) ? (mw[j >> 1] & 0xffffu) | (m << 16) : (mw[j >> 1] & 0xffff0000u) | m;
                }
        put_magphase(y, full, u32x4{mw[0], mw[1], mw[2], mw[3]}, u32x2{pw[0], pw[1]});
    }

    // ScaleImage to (w/2, h/2), rows y and y+1 (y even).  With xscale = yscale = 2 the reference's fixed-point
    // setup (xinc = 2^19, xoffs = 2^17) gives source column 2x and row 2y with weight 128 on both pixels, so the
    // two-stage SIMD rule is ((p00+p01+1)>>1 + (p10+p11+1)>>1 + 1) >> 1 -- rounded byte means, v_lerp_u8 -- and the
    // single-rounding tail (columns >= (w/2) & ~7) is (p00+p01+p10+p11+2) >> 2; the row and column clamps never
    // engage.
    MVX_DEV void half(int y, const RawRow &a, const RawRow &b) const
    {
        const int dw = w >> 1, xh = x >> 1;
        const long ph = (long)(y >> 1) * d.halfStride + xh;
        if (xh + 4 <= (dw & ~7)) {
            uint32_t m[2];
#pragma unroll
            for (int k = 0; k < 2; k++)   // bytes 0 and 2
                m[k] = __builtin_amdgcn_lerp(__builtin_amdgcn_lerp(a.w[k], a.w[k] >> 8, 0x01010101u),
                                             __builtin_amdgcn_lerp(b.w[k], b.w[k] >> 8, 0x01010101u), 0x01010101u);
            *at<uint32_t>(d.half, ph) = __builtin_amdgcn_perm(m[1], m[0], 0x06040200u);
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int sh = 16 * (j & 1);
            const uint32_t p = a.w[j >> 1] >> sh, q = b.w[j >> 1] >> sh;
            if (xh + j < dw) *at<uint8_t>(d.half, ph + j) = (uint8_t)(((p & 0xffu) + ((p >> 8) & 0xffu) + (q & 0xffu) + ((q >> 8) & 0xffu) + 2) >> 2);
        }
    }
};

// `units` waves' worth of tiles
template <int TW>
__global__ void __launch_bounds__(CHAIN_THREADS)
k_chain_batch(const ChainRow *__restrict__ plan, uint32_t count, uint32_t units)
{
    constexpr uint32_t LPT = TW / 8, TPW = 64 / LPT;   // lanes per tile, tiles per wave
    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, step = (gridDim.x >> 3) * (CHAIN_THREADS / 64);
    const uint32_t span = (units + 7u) / 8u;
    const uint32_t uBegin = xcd * span, uEnd = min(units, uBegin + span);
    for (uint32_t u = uBegin + slot * (CHAIN_THREADS / 64) + wave; u < uEnd; u += step) {
        const ChainRow &d = plan[find_image(plan, count, u * TPW)];
        const uint32_t rows = d.rows;
        const uint32_t tile = u * TPW - d.tileBegin + lane / LPT, ty = tile / d.tilesX, tx = tile - ty * d.tilesX;
        const int x = (int)(tx * TW + 8 * (lane % LPT)), y0 = (int)(ty * rows);
        const int w = (int)d.w, h = (int)d.h, stride = (int)d.srcStride;
        if (x >= w || y0 >= h) continue;
        ChainLane L{d, w, h, stride, h * stride, x};
        uint32_t two = 0x00020002u;
        asm("" : "+s"(two));
        L.two = pair_of(two);
        L.merged = d.gx == nullptr;
        L.wrapL = stride == w;
        L.rightOk = x + 8 < w;
        L.wrapR = x + 8 == stride;
        L.edge = x == 0 || !L.rightOk || y0 < 2 || y0 + (int)rows > h - 2;
#pragma unroll
        for (int k = 0; k < 2; k++) {   // (widths are even: a pair's columns c, c+2 end at w - c > 0, > 2)
            const int e = x + 4 * k, o = e + 1;
            L.colE[k] = (e < w ? 0xffffu : 0u) | (e + 2 < w ? 0xffff0000u : 0u);
            L.colO[k] = (o < w ? 0xffffu : 0u) | (o + 2 < w ? 0xffff0000u : 0u);
        }
        const bool wantHalf = d.half != nullptr;
        const auto split = [](const u32x4 &v) {
            InRow r;
#pragma unroll
            for (int k = 0; k < 4; k++) { r.E[k] = even_bytes(v[k]); r.O[k] = odd_bytes(v[k]); }
            return r;
        };
        // Step k takes input row y0+k (next), which completes blurred row y0+k-1 and, from k = 2 on, output row
        // y0+k-2.  Two rows of each kind are kept and the new one goes over the older, so the caller swaps the
        // arguments instead of the values.
        InRow ia = split(L.load(y0 - 2)), ib = split(L.load(y0 - 1));
        u32x4 next = L.load(y0);
        BlurRow ba{}, bb{};
        RawRow ra{}, rb{};
        const auto row = [&](int k, InRow &iO, InRow &iN, BlurRow &bO, BlurRow &bN, RawRow &rO, RawRow &rN) {
            const u32x4 cur = next;
            next = L.load(y0 + k + 1);
            const InRow in = split(cur);
            const BlurRow b = L.blur(y0 + k - 1, iO, iN, in);
            if (k >= 2 && y0 + k - 2 < h) {
                L.gradients(y0 + k - 2, bO, bN, b);
                if (wantHalf && !(k & 1)) L.half(y0 + k - 2, rO, rN);
            }
            iO = in;
            bO = b;
            rO.w[0] = cur[1];
            rO.w[1] = cur[2];
        };
#pragma unroll 1
        for (int k = 0; k < (int)rows + 2; k += 2) {
            row(k, ia, ib, ba, bb, ra, rb);
            row(k + 1, ib, ia, bb, ba, rb, ra);
        }
    }
}

// ------------------------------------------------------------------ host side ------------------
struct TileShape { int tw, th; };
constexpr TileShape kShapes[MVX_CHAIN_TILE_COUNT] = {{16, 16}, {32, 16}, {32, 32}, {64, 16}, {64, 32}};

typedef void (*ChainKernel)(const ChainRow *, uint32_t, uint32_t);
constexpr ChainKernel kKernels[MVX_CHAIN_TILE_COUNT] = {k_chain_batch<16>, k_chain_batch<32>, k_chain_batch<32>, k_chain_batch<64>,
                                                        k_chain_batch<64>};
// tiles one wave takes side by side
constexpr uint32_t tiles_per_wave(uint32_t tile) { return 64u / ((uint32_t)kShapes[tile].tw / 8u); }

// an image's waves with tiles of `rows` rows
inline uint64_t image_waves(uint32_t w, uint32_t h, uint32_t rows, uint32_t tile)
{
    const uint32_t tw = (uint32_t)kShapes[tile].tw, per = tiles_per_wave(tile);
    return ((uint64_t)((w + tw - 1) / tw) * ((h + rows - 1) / rows) + per - 1) / per;
}

// Rows a lane streams at most: the tile shape's, halved down to 2 while the whole batch (`waves` of tiles of the
// shape's height) is fewer than 8192 waves (eight for each of
// the 1024 SIMDs, of which about four run at a time, so that no SIMD ends long after the others: 48 uneven images with
// 64x32 tiles took 294 us at 2048, 283 at 8192); a lane's rows cost one more load and blur above and below them each.
// A small batch is bound by the chain of a lane's rows, each a wait for memory: one 320x240 image 9.8 us with no fewer
// than 4 rows, 6.7 with 2, 4096x2160 10.6 and 9.0.
inline uint32_t batch_rows(uint64_t waves, uint32_t tile)
{
    uint32_t rows = (uint32_t)kShapes[tile].th;
    while (rows > 2 && waves < 8192) { rows /= 2; waves *= 2; }
    return rows;
}

// Rows a lane streams of one image: of those up to the batch's the ones with the least work, a wave's being its rows
// and the four more that it loads.  An image much smaller than a wave of tiles so gets more, lower ones that fill
// the wave's lanes (64x32 tiles: 4096 images of 64x64 36 us, 112 with all at the batch's rows; 1024 of them 14 and 36).
inline uint32_t image_rows(uint32_t w, uint32_t h, uint32_t most, uint32_t tile)
{
    uint32_t best = most;
    uint64_t least = image_waves(w, h, most, tile) * (most + 4);
    for (uint32_t rows = most / 2; rows >= 2; rows /= 2) {
        const uint64_t work = image_waves(w, h, rows, tile) * (rows + 4);
        if (work < least) { least = work; best = rows; }
    }
    return best;
}

inline bool plane_ok_cb(const void *p, uint32_t w, uint32_t stride, uint32_t bpp)
{
    return p && aligned16(p) && (stride % 16u) == 0 && stride >= ((w * bpp + 15u) & ~15u);
}

bool image_ok(const mvx_chain_image_t &im)
{
    const uint32_t w = im.width, h = im.height;
    if (w < 2 || h < 2 || (w & 1u) || (h & 1u) || w > 65536u || h > 65536u) return false;
    if ((uint64_t)h * im.srcStride >= (1ull << 31)) return false;
    // gx and gy: both stored, or both NULL (virtual gradients, merged rules)
    const bool merged = !im.gx && !im.gy;
    if (!plane_ok_cb(im.src, w, im.srcStride, 1) || (!merged && (!plane_ok_cb(im.gx, w, im.gxStride, 2) ||
        !plane_ok_cb(im.gy, w, im.gyStride, 2))) || !plane_ok_cb(im.mag, w, im.magStride, 2) ||
        !plane_ok_cb(im.phase, w, im.phaseStride, 1))
        return false;
    if (im.half && !plane_ok_cb(im.half, w / 2, im.halfStride, 1)) return false;
    return true;
}

int device_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return cus;
}

}  // namespace mvx

using namespace mvx;

extern "C" size_t mvx_ChainBatch_workspace_size(uint32_t count) { return (size_t)count * sizeof(ChainRow); }

// batchPD front end: image i of every tall plane starts at row i * (the plane's rows per image)
extern "C" int mvx_ChainBatch_prepare_batchPD(const uint8_t *src, uint32_t srcStride, uint32_t maxHeight, const uint32_t *widths,
                                              const uint32_t *heights, uint32_t nbatch, int16_t *gx, uint32_t gxStride, int16_t *gy,
                                              uint32_t gyStride, int16_t *mag, uint32_t magStride, uint8_t *phase,
                                              uint32_t phaseStride, uint8_t *half, uint32_t halfStride, uint32_t halfMaxHeight,
                                              uint32_t tile, uint32_t workgroupsPerCU, void *workspace, size_t workspaceSize,
                                              mvx_chain_plan_t *plan)
{
    if (!src || !widths || !heights || nbatch == 0 || !gx != !gy || !mag || !phase || !plan) return MVX_ERROR_INVALID_PARAMETERS;
    std::vector<mvx_chain_image_t> images(nbatch);
    for (uint32_t i = 0; i < nbatch; i++) {
        if (heights[i] > maxHeight || (half && heights[i] / 2 > halfMaxHeight)) return MVX_ERROR_INVALID_PARAMETERS;
        mvx_chain_image_t &im = images[i];
        im.src = src + (size_t)i * maxHeight * srcStride;
        im.width = widths[i];
        im.height = heights[i];
        im.srcStride = srcStride;
        im.gx = gx ? (int16_t *)((uint8_t *)gx + (size_t)i * maxHeight * gxStride) : nullptr;
        im.gxStride = gxStride;
        im.gy = gy ? (int16_t *)((uint8_t *)gy + (size_t)i * maxHeight * gyStride) : nullptr;
        im.gyStride = gyStride;
        im.mag = (int16_t *)((uint8_t *)mag + (size_t)i * maxHeight * magStride);
        im.magStride = magStride;
        im.phase = phase + (size_t)i * maxHeight * phaseStride;
        im.phaseStride = phaseStride;
        im.half = half ? half + (size_t)i * halfMaxHeight * halfStride : nullptr;
        im.halfStride = halfStride;
    }
    return mvx_ChainBatch_prepare(images.data(), nbatch, tile, workgroupsPerCU, workspace, workspaceSize, plan);
}

extern "C" int mvx_ChainBatch_prepare(const mvx_chain_image_t *images, uint32_t count, uint32_t tile,
                                      uint32_t workgroupsPerCU, void *workspace, size_t workspaceSize,
                                      mvx_chain_plan_t *plan)
{
    if (!images || !plan || count == 0 || tile >= MVX_CHAIN_TILE_COUNT || !workspace || !aligned16(workspace) ||
        workspaceSize < mvx_ChainBatch_workspace_size(count))
        return MVX_ERROR_INVALID_PARAMETERS;
    const TileShape s = kShapes[tile];
    std::vector<ChainRow> rows(count);
    uint64_t waves = 0;
    for (uint32_t i = 0; i < count; i++) {
        if (!image_ok(images[i])) return MVX_ERROR_INVALID_PARAMETERS;
        waves += image_waves(images[i].width, images[i].height, (uint32_t)s.th, tile);
    }
    const uint32_t most = batch_rows(waves, tile);
    uint64_t tiles = 0;
    for (uint32_t i = 0; i < count; i++) {
        const mvx_chain_image_t &im = images[i];
        ChainRow &r = rows[i];
        std::memset(&r, 0, sizeof(r));
        r.src = im.src; r.gx = im.gx; r.gy = im.gy; r.mag = im.mag; r.phase = im.phase; r.half = im.half;
        r.w = im.width; r.h = im.height;
        r.srcStride = im.srcStride; r.gxStride = im.gxStride; r.gyStride = im.gyStride;
        r.magStride = im.magStride; r.phaseStride = im.phaseStride; r.halfStride = im.halfStride;
        r.tilesX = (im.width + s.tw - 1) / s.tw;
        r.tileBegin = (uint32_t)tiles;
        r.rows = image_rows(im.width, im.height, most, tile);
        tiles += image_waves(im.width, im.height, r.rows, tile) * tiles_per_wave(tile);   // a wave's lanes share one image
        if (tiles >= (1ull << 31)) return MVX_ERROR_INVALID_PARAMETERS;
    }
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void *>(kKernels[tile]), CHAIN_THREADS, 0) !=
            hipSuccess || occ <= 0)
        return MVX_FAILURE;
    const int cus = device_cus();
    if (cus <= 0) return MVX_FAILURE;
    const uint32_t perCu = workgroupsPerCU == 0 ? (uint32_t)occ : std::min<uint32_t>(workgroupsPerCU, (uint32_t)occ);
    uint32_t wgs = (uint32_t)cus * perCu;
    // no more workgroups than there are waves' units for (rounded to a multiple of the 8 XCDs)
    const uint64_t units = tiles / tiles_per_wave(tile);
    const uint64_t perXcd = ((units + 7) / 8 + CHAIN_THREADS / 64 - 1) / (CHAIN_THREADS / 64);
    wgs = (uint32_t)std::min<uint64_t>(wgs, perXcd * 8);
    wgs = std::max<uint32_t>(8u, wgs & ~7u);
    if (hipMemcpy(workspace, rows.data(), rows.size() * sizeof(ChainRow), hipMemcpyHostToDevice) != hipSuccess)
        return MVX_FAILURE;
    plan->table = workspace;
    plan->count = count;
    plan->numTiles = (uint32_t)tiles;
    plan->tile = tile;
    plan->workgroups = wgs;
    plan->tileWidth = (uint32_t)s.tw;
    plan->tileHeight = (uint32_t)s.th;
    return MVX_SUCCESS;
}

extern "C" int mvx_ChainBatch_run(mvx_stream_t stream, const mvx_chain_plan_t *plan)
{
    if (!plan || !plan->table || plan->tile >= MVX_CHAIN_TILE_COUNT || plan->count == 0 || plan->workgroups < 8 ||
        (plan->workgroups & 7u))
        return MVX_ERROR_INVALID_PARAMETERS;
    if (plan->numTiles == 0) return MVX_SUCCESS;
    hipLaunchKernelGGL(kKernels[plan->tile], dim3(plan->workgroups), dim3(CHAIN_THREADS), 0, stream_of(stream),
                       (const ChainRow *)plan->table, plan->count, plan->numTiles / tiles_per_wave(plan->tile));
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" int mvx_ChainBatch_autotune(mvx_stream_t stream, const mvx_chain_image_t *images, uint32_t count,
                                       uint32_t reps, void *workspace, size_t workspaceSize, mvx_chain_plan_t *best,
                                       float *msTable)
{
    if (!best || reps == 0) return MVX_ERROR_INVALID_PARAMETERS;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return MVX_FAILURE;
    if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); return MVX_FAILURE; }
    static const uint32_t kPerCu[MVX_CHAIN_OCCUPANCY_STEPS] = {1, 2, 4, 0};  // 0 = the occupancy limit
    float bestMs = -1.f;
    uint32_t bestTile = 0, bestPerCu = 0;
    int rc = MVX_SUCCESS;
    for (uint32_t tile = 0; tile < MVX_CHAIN_TILE_COUNT && rc == MVX_SUCCESS; tile++) {
        for (int o = 0; o < MVX_CHAIN_OCCUPANCY_STEPS && rc == MVX_SUCCESS; o++) {
            mvx_chain_plan_t p;
            rc = mvx_ChainBatch_prepare(images, count, tile, kPerCu[o], workspace, workspaceSize, &p);
            if (rc != MVX_SUCCESS) break;
            rc = mvx_ChainBatch_run(stream, &p);  // warm-up
            if (rc != MVX_SUCCESS) break;
            (void)hipEventRecord(e0, stream_of(stream));
            for (uint32_t k = 0; k < reps && rc == MVX_SUCCESS; k++) rc = mvx_ChainBatch_run(stream, &p);
            (void)hipEventRecord(e1, stream_of(stream));
            if (hipEventSynchronize(e1) != hipSuccess) { rc = MVX_FAILURE; break; }
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            ms /= (float)reps;
            if (msTable) msTable[tile * MVX_CHAIN_OCCUPANCY_STEPS + o] = ms;
            if (bestMs < 0.f || ms < bestMs) { bestMs = ms; bestTile = tile; bestPerCu = kPerCu[o]; }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != MVX_SUCCESS) return rc;
    // leave the workspace holding the winner's table
    return mvx_ChainBatch_prepare(images, count, bestTile, bestPerCu, workspace, workspaceSize, best);
}

extern "C" int mvx_ChainBatch_graph_create(const mvx_chain_plan_t *plan, void **graphExec)
{
    if (!plan || !graphExec) return MVX_ERROR_INVALID_PARAMETERS;
    *graphExec = nullptr;
    hipStream_t s = nullptr;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return MVX_FAILURE;
    hipGraph_t g = nullptr;
    hipGraphExec_t e = nullptr;
    int rc = MVX_FAILURE;
    if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess) {
        const int launched = mvx_ChainBatch_run(s, plan);
        const hipError_t ended = hipStreamEndCapture(s, &g);
        if (launched == MVX_SUCCESS && ended == hipSuccess && g &&
            hipGraphInstantiate(&e, g, nullptr, nullptr, 0) == hipSuccess) {
            *graphExec = e;
            rc = MVX_SUCCESS;
        } else if (launched != MVX_SUCCESS) {
            rc = launched;
        }
    }
    if (g) (void)hipGraphDestroy(g);
    (void)hipStreamDestroy(s);
    return rc;
}

extern "C" int mvx_graph_launch(void *graphExec, mvx_stream_t stream)
{
    if (!graphExec) return MVX_ERROR_INVALID_PARAMETERS;
    return hipGraphLaunch(reinterpret_cast<hipGraphExec_t>(graphExec), stream_of(stream)) == hipSuccess ? MVX_SUCCESS
                                                                                                       : MVX_FAILURE;
}

extern "C" int mvx_graph_destroy(void *graphExec)
{
    if (!graphExec) return MVX_SUCCESS;
    return hipGraphExecDestroy(reinterpret_cast<hipGraphExec_t>(graphExec)) == hipSuccess ? MVX_SUCCESS : MVX_FAILURE;
}
