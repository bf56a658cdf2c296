// vision_graph.hip -- the RGB vision graph as a few fused, frame-batched launches for gfx950.
//
// Graph (the reference schedules ~15 kernels per frame for it, with host round trips for the Canny
// trace and the Harris pick):
//   RGB -> ColorConvert Y (virtual) -> { ChannelCopy -> pyramid level 0,
//                                         ScaleImage 2:1 bilinear,
//                                         ScaleGaussianHalf_5x5 -> pyramid levels 1..,
//                                         Canny 3x3 L1 (Sobel -> NMS/threshold -> hysteresis),
//                                         Harris 3x3/3x3 (HG3 -> score -> NMS -> sort and pick) }
//
// Launches per batch of frames (blockIdx.z = frame):
//   k_front     one 58x32 luma tile (+3 halo) per wave, four independent waves per workgroup.  Every
//               window row of the tile (64 luma, 62 gradient, 60 score columns) fits the 64 lanes, so
//               lane = column and the wave streams the tile's rows top to bottom with every quantity in
//               rolling register windows (column neighbours through DPP lane shifts): RGB -> Y, level 0,
//               the 2:1 scaled image, level 1, Canny gradients/NMS/threshold, Harris products / exact
//               integer window sums / score / NMS; then tile-local hysteresis on 64-bit row masks
//               (lane = row) with the border-touching weak components labelled by flood fill.  No
//               barriers; LDS holds only the wave's Harris candidates.  Only graph outputs and small
//               per-tile tables reach HBM.  Tiles away from the image border take a branch-free
//               instantiation.
//   k_border    unions the hysteresis components that touch tile borders, across tiles.  Strong
//               components get ids below every weak one, so after atomicMin linking a set's root is
//               strong iff the set holds a strong component -- no marking pass.
//   k_resolve   the undecided weak pixels k_front listed per tile take their global root's state.
//   k_half      pyramid levels 2.. (one launch per level, all frames).
//   k_pick      Harris sort and pick, one workgroup per frame (pick.hpp).
//
// Every output is bit-exact with the reference CPU path; the equivalences used are stated where they
// are used.  Limits of the fused path (callers use the per-node kernels otherwise): width >= 16 and a
// multiple of 4 (the HG3 pitch quirk is then the identity), even height, scaled image exactly half
// size, every pyramid step one the reference accepts.
#include "mvx_common.hpp"
#include "pick.hpp"
#include "rowmask.hpp"
#include "pyramid.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

namespace mvx {

constexpr int TW = 58, TH = 32;                  // luma tile
constexpr int HY = 3;                            // luma halo: Sobel 1 + Harris window 1 + NMS 1
constexpr int TP = 64;                           // row pitch of pixel indices in a tile (one wave row)
constexpr int YH = TH + 2 * HY;                  // luma window rows (columns: TW + 6 = 64)
constexpr int TS = TH * TP;                      // tile-local pixel index space, p = ly * TP + lx
constexpr int TNB = 2 * (TW + TH);               // union-find slots per tile: one per border pixel, at most

struct FrameDesc {
    const uint8_t *rgb; uint32_t rgbStride;
    uint8_t *lvl[8]; uint32_t lvlStride[8];      // pyramid levels, lvl[0] = luma
    uint8_t *scaled; uint32_t scaledStride;
    uint8_t *edges; uint32_t edgesStride;
    void *corners; uint32_t *numItems; uint64_t *count;
    // per-frame workspace
    int32_t *border;      // tiles x 2(TW+TH) component ids of tile-border pixels (-1: none)
    uint32_t *parent;     // 1 + tiles * TNB union-find slots: 0 the strong node, then TNB per tile
    uint32_t *ulist;      // tiles x TS: a tile's undecided pixels, p | the component's number k << 16
    uint32_t *ucount;     // tiles: undecided pixels listed
    void *cand;           // Harris XYS candidates
    uint32_t *candCount;  // candidates appended (reset by k_pick)
    void *pickWs;         // harris pick workspace
};

struct GraphParams {
    int w, h, yStride, tilesX, tilesY;
    int dw, dh;            // scaled size (w/2, h/2)
    int levels;
    int lvlW[8], lvlH[8];
    uint32_t lower, upper;
    float k, thr, norm, dist;
    float normRcp;           // RN(1 / norm)
    float hotMc;             // a score above thr needs mc > hotMc (and, k >= 0, gx2 * gy2 > hotProd)
    float hotProd;
    int upperBits, lowerBits;      // the Canny thresholds as float bits, magnitudes being float bits too
    uint64_t upperAll, lowerAll;   // all ones where a threshold is negative as an int (every pixel above it)
    uint32_t capacity, candCap;
};

// luma of one RGB pixel, HafCpu_ColorConvert_Y_RGB (ago_haf_cpu_color_convert.cpp:2913-2990):
// ((R * 0.2126f) + G * 0.7152f) + B * 0.0722f in float, truncated, saturated
template <class Ptr> MVX_DEV uint32_t luma(Ptr p)
{
    float v = (float)p[0] * 0.2126f;
    v = v + (float)p[1] * 0.7152f;
    v = v + (float)p[2] * 0.0722f;
    const int iv = (int)v;
    return (uint32_t)min(max(iv, 0), 255);
}

// four bytes at any address
struct __attribute__((packed, aligned(1))) RgbDword { uint32_t v; };

// the virtual luma plane at linear position (r, c): stride yStride, padding and guard bytes zero
MVX_DEV uint32_t yflat(const FrameDesc &F, const GraphParams &P, int r, int c)
{
    if (c >= 0 && c < P.w && r >= 0 && r < P.h) return luma(gmem(F.rgb) + (long)r * F.rgbStride + 3L * c);
    const long i = (long)r * P.yStride + c;
    if (i < 0 || i >= (long)P.h * P.yStride) return 0;
    r = (int)(i / P.yStride);
    c = (int)(i - (long)r * P.yStride);
    if (c >= P.w) return 0;
    return luma(gmem(F.rgb) + (long)r * F.rgbStride + 3L * c);
}

// the value of lane + 1 of the wave (DPP wave_shl:1; lane 63 reads 0)
MVX_DEV int lane_next(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }

MVX_DEV float lane_next_f(float v) { return __int_as_float(lane_next(__float_as_int(v))); }

// lane masks: one compare gives one (no VALU work beyond it), and masks combine, shift and wait in scalar
// registers
MVX_DEV uint64_t mask_of(bool v) { return __builtin_amdgcn_ballot_w64(v); }
MVX_DEV bool in_mask(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
extern "C" __device__ int mvx_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

constexpr int FTW = 4;                                     // tiles (one wave each) per workgroup of k_front
constexpr int RES_TILES = 4;                               // tiles per wave of k_resolve
constexpr int CAND_MAX = ((TW + 1) / 2) * ((TH + 1) / 2);  // Harris NMS maxima of a tile are never 8-adjacent

// One wave streams one tile: luma window rows k = 0..YH-1 (image row ty0-3+k, lane = column tx0-3+lane)
// top to bottom, every later quantity from rolling register windows of the rows it needs, column
// neighbours by DPP lane shifts.  At step k:
//   luma row k -> pyramid level 0 (row k-3), the 2:1 scaled image and level 1 when their rows complete;
//   gradient row (image row ty0+k-4, column tx0-2+lane) -> Canny magnitude and sector masks, HG3 products
//   and 3-column sums;
//   Canny NMS and double threshold of tile row k-5 into 64-bit row masks (edge, strong; lane r holds row r);
//   Harris score row (image row ty0+k-5, column tx0-1+lane), Harris NMS of tile row k-6 into the per-wave
//   candidate buffer.
// Then the tile's hysteresis on the row masks and the settle pass.
//
// Bound by VALU issue, so the instructions of a row are what counts (16 frames of 3840x2160: 690 us with
// about 125 of them, 505 us with about 68):
//   * luma, gradients, products and window sums are floats holding integers below 2^24 -- exact, like the
//     integers the reference computes -- so the Canny sector test, the Harris score and |.| need no
//     conversions; a 16-bit integer form exists for none of the float rules;
//   * a pixel's Canny sector is never stored: its three compares leave lane masks in scalar registers, which
//     wait there for the next row and select the NMS neighbours from there;
//   * Harris scores above the threshold are rare, so a row first asks whether any lane can have one
//     (gx2 * gy2 > thr * norm, then mc > thr * norm: scalar branches), and only then divides, compares
//     and suppresses.
template <bool INNER>
MVX_DEV void front_tile(uint64_t *cand, const FrameDesc &F, const GraphParams &P, int tx0, int ty0, int tile)
{
    const int lane = (int)threadIdx.x & 63;
    const int w = P.w, h = P.h;
    const int tw = INNER ? TW : min(TW, w - tx0), th = INNER ? TH : min(TH, h - ty0);
    const int x = tx0 - 1 + lane;       // Canny magnitude / Harris score column
    const int ox = tx0 + lane;          // tile output column

    // inner tiles read a pixel's R, G, B (and the next pixel's R) with one dword load; the window's
    // last column is at most w-2, so the dword stays inside the row
    const __amdgpu_buffer_rsrc_t rgbR = plane_rsrc(F.rgb), l0R = plane_rsrc(F.lvl[0]), scR = plane_rsrc(F.scaled);
    const __amdgpu_buffer_rsrc_t l1R = plane_rsrc(F.lvl[1]);
    const uint32_t rgbStride = F.rgbStride, l0Stride = F.lvlStride[0], l1Stride = F.lvlStride[1], scStride = F.scaledStride;
    const int rgbCol = 3 * (tx0 - HY + lane);
    // other tiles read the virtual luma plane at linear addresses: a column before 0 or past the stride lies in
    // the row above or below (edgeRow), one of the padding or outside the plane is 0.  The same dword loads,
    // two rows ahead, from a row clamped into the image; the last column's dword starts one byte early.
    // Images narrower than a tile's window may wrap more than once: they go through yflat.
    const bool wide = w >= 64;
    const uint64_t rgbAddr = (uint64_t)F.rgb;
    int edgeRow = 0, edgeCol = tx0 - HY + lane;
    if (edgeCol < 0) { edgeRow = -1; edgeCol += P.yStride; }
    else if (edgeCol >= P.yStride) { edgeRow = 1; edgeCol -= P.yStride; }
    const bool edgeColOk = edgeCol < w;
    const uint32_t edgeOff = edgeColOk ? 3u * (uint32_t)edgeCol - (edgeCol == w - 1 ? 1u : 0u) : 0u, edgeShift = edgeCol == w - 1 ? 8u : 0u;
    auto fetch = [&](int k) -> uint32_t {
        if (INNER) return __builtin_amdgcn_raw_buffer_load_b32(rgbR, rgbCol, (int)((uint32_t)(ty0 - HY + k) * rgbStride), 0);
        // 64-bit row addresses, since a frame can be a narrow view of a wide buffer; the three that a lane chooses
        // from are scalar arithmetic
        const auto row = [&](int r) { return rgbAddr + (uint64_t)(uint32_t)min(max(r, 0), h - 1) * rgbStride; };
        const int r = ty0 - HY + k;
        const uint64_t above = row(r - 1), same = row(r), below = row(r + 1);
        return ((gptr_t<const RgbDword>)((edgeRow < 0 ? above : edgeRow > 0 ? below : same) + edgeOff))->v;
    };
    // luma row k from its fetched dwords
    auto luma_of = [&](int k, uint32_t p) -> int {
        if (!INNER) p >>= edgeShift;
        float f = (float)(p & 0xffu) * 0.2126f;
        f = f + (float)((p >> 8) & 0xffu) * 0.7152f;
        f = f + (float)((p >> 16) & 0xffu) * 0.0722f;
        const int v = (int)f;
        if (INNER) return v;
        const int r = ty0 - HY + k + edgeRow;
        return edgeColOk && r >= 0 && r < h ? v : 0;
    };
    const int body = P.dw & ~7;
    const int oxp = (w & 1) ? 0 : 1, oyp = (h & 1) ? 0 : 1;
    // Harris scores compare as int32 keys: a non-negative float's bits order like the float; with a
    // negative threshold negative scores occur, and the key flips their magnitude bits (an involution).
    // Scores are never -0 (mc is never -0), so equal keys are equal scores.
    const bool negKeys = P.thr < 0.0f;
    // output columns of this lane: level 0 (luma lane), 2:1 scaled (lane 2X'+3), level 1 (lane 2X'+oxp+1)
    const int sp = lane - HY, lp1 = lane - oxp - 1;
    const bool scOut = sp >= 0 && !(sp & 1) && (sp >> 1) < TW / 2 && tx0 / 2 + (sp >> 1) < P.dw;
    const bool l1Out = lp1 >= 0 && !(lp1 & 1) && (lp1 >> 1) < TW / 2 && tx0 / 2 + (lp1 >> 1) < P.lvlW[1];
    const bool allBody = tx0 / 2 + TW / 2 <= body;         // no column of the scaled image's scalar tail
    const bool scBody = tx0 / 2 + (sp >> 1) < body;
    const uint64_t outCols = INNER ? (1ull << TW) - 1 : mask_of(lane < TW && ox >= 1 && ox <= w - 2);

    int emLo = 0, emHi = 0, smLo = 0, smHi = 0;           // lane r: edge / strong mask of tile row r
    uint32_t nc = 0;                                      // candidates in the wave's buffer
    uint64_t sec0 = 0, sec2 = 0, sec3 = 0;                // sector tests of the Canny centre row (see below)
    int aPrev = 0;                                        // 2:1 scaled: rounded pair means of luma row k-1
    float tPrev = 0.0f;                                   // luma pair sums of row k-1
    int Vb = 0;                                           // Harris score key row k-5
    bool hotB = false;                                    // ... has a lane with a score

    // One step of the stream (luma row k).  Windows deeper than one row are passed in age order and
    // the step writes its new row over the oldest one, so the caller rotates the arguments instead of
    // the values (no register copies): yA..yD = luma rows k-4..k-1 (yA <- row k); dO, dN / sO, sN = rows
    // k-2, k-1 (dO <- row k); xx0.. = HG3 sums of the two gradient rows above (<- this row's); uO, uN / vO, vN =
    // the two magnitude rows above at columns tx0-1+lane and tx0+lane (<- this row's); HO, HN = score key
    // 3-column maxima rows k-6, k-5 (HO <- row k-4); pO, pN = RGB of rows k, k+1 (pO <- row k+2).
    auto step = [&](const int k, uint32_t &pO, uint32_t &pN, float &yA, float &yB, float &yC, float &yD, float &dO,
                    float &dN, float &sO, float &sN, float &xx0, float &xx1, float &xy0, float &xy1, float &yy0,
                    float &yy1, int &uO, int &uN, int &vO, int &vN, int &HO, int &HN) {
        // ---- luma row k (ColorConvert Y of the RGB pixel, or the virtual plane's linear-address
        //      value); the float sum lies in [0, 256), so the truncation needs no clamp
        int yi;
        if (INNER || wide) {
            const uint32_t cur = pO;
            if (k + 2 < YH) pO = fetch(k + 2);
            yi = luma_of(k, cur);
        } else {
            yi = (int)yflat(F, P, ty0 - HY + k, tx0 - HY + lane);
        }
        const float yk = (float)yi;
        if (k >= HY && k < HY + th && lane >= HY && lane < HY + tw)
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)yi, l0R, tx0 - HY + lane, (int)((uint32_t)(ty0 + k - HY) * l0Stride), 0);
        // binomial column sums through one-lane shifts: t = Y[l]+Y[l+1], s = Y[l]+2Y[l+1]+Y[l+2], d = Y[l+2]-Y[l]
        const float tk = yk + lane_next_f(yk);
        const float sk = tk + lane_next_f(tk), dk = lane_next_f(tk) - tk;

        // ---- ScaleImage 2:1 (ago_haf_cpu_geometric.cpp:2000-2045 with xscale = yscale = 2, offsets 0.5):
        //      output row oy from luma rows 2oy+3 (k-1) and 2oy+4 (k); lane 2X'+3 holds output column X'.
        //      The body rounds twice -- (128 a + 128 b + 0x80) >> 8 is the rounded mean of two bytes, one
        //      v_lerp_u8 --, the scalar tail once: (128 * 128 sum + 0x8000) >> 16
        const int ak = (int)__builtin_amdgcn_lerp((uint32_t)yi, (uint32_t)lane_next(yi), 1u);
        if (k >= 4 && !(k & 1) && k <= HY + TH - 1) {
            const int Yo = ty0 / 2 + ((k - 4) >> 1);
            int v = (int)__builtin_amdgcn_lerp((uint32_t)aPrev, (uint32_t)ak, 1u);
            if (!allBody) v = scBody ? v : ((int)(tPrev + tk) + 2) >> 2;
            if (Yo < P.dh && scOut)
                __builtin_amdgcn_raw_buffer_store_b8((uint8_t)v, scR, tx0 / 2 + (sp >> 1), (int)((uint32_t)Yo * scStride), 0);
        }
        aPrev = ak;
        tPrev = tk;
        // ---- ScaleGaussianHalf_5x5 level 1 (ago_haf_cpu_pyramid.cpp:94-305): centre (2X+oxp, 2Y+oyp),
        //      luma rows k-4..k; the horizontal 1 4 6 4 1 is four "v + v[l+1]" steps, so lane 2X'+oxp+1
        //      holds the sum over columns lane..lane+4 (centre lane+2); at most 255 * 256
        if (P.levels > 1 && k >= 5 + oyp && !((k - 5 - oyp) & 1)) {
            const int oy = (k - 5 - oyp) >> 1, Yo = ty0 / 2 + oy;
            if (oy < TH / 2 && Yo >= 1 && Yo <= P.lvlH[1] - 2) {
                float acc = fmaf(6.0f, yC, fmaf(4.0f, yB + yD, yA + yk));
                acc = acc + lane_next_f(acc);
                acc = acc + lane_next_f(acc);
                acc = acc + lane_next_f(acc);
                acc = acc + lane_next_f(acc);
                if (l1Out)
                    __builtin_amdgcn_raw_buffer_store_b8((uint8_t)((uint32_t)acc >> 8), l1R, tx0 / 2 + (lp1 >> 1),
                                                         (int)((uint32_t)Yo * l1Stride), 0);
            }
        }

        // ---- Sobel gradient row (linear-address luma; |gx|, |gy| <= 1020, so the reference's S16 values are
        //      these), HG3 products and 3-column sums.  HG3 rows 0 and h-1 are never written (zero).  The
        //      9-sums of products stay below 2^24, so every sum here is exact in any order.
        const int yg = ty0 + k - 4;
        const float gx = fmaf(2.0f, dN, dO) + dk, gy = sk - sO;
        float pxx = gx * gx, pxy = gx * gy, pyy = gy * gy;
        if (!INNER && (yg < 1 || yg > h - 2)) pxx = pxy = pyy = 0.0f;
        const float hxx = pxx + lane_next_f(pxx + lane_next_f(pxx));
        const float hxy = pxy + lane_next_f(pxy + lane_next_f(pxy));
        const float hyy = pyy + lane_next_f(pyy + lane_next_f(pyy));

        // ---- Harris score row k-4 (image row ty0+k-5): Vc = mc / norm > T ? mc / norm : 0, the quotient exactly
        //      the IEEE one; kept as its compare key, with the maximum of the key over columns lane..lane+2
        int Vc = 0, Hc = 0;
        bool hot = false;
        {
            const int yv = ty0 + k - 5;
            const float gx2 = (xx0 + xx1) + hxx, gy2 = (yy0 + yy1) + hyy;
            const float prod = gx2 * gy2;
            if (k >= 4 && mask_of(prod > P.hotProd)) {
                const float gxy2 = (xy0 + xy1) + hxy;
                const float tr = gx2 + gy2;
                const float det = prod - (gxy2 * gxy2);
                const float mc = det - (P.k * tr * tr);
                if (mask_of(mc > P.hotMc)) {
                    const float q = div_by_const_rn(mc, P.norm, P.normRcp);
                    float v = (q > P.thr) ? q : 0.0f;
                    if (!INNER && !(x >= 1 && x <= w - 2 && yv >= 1 && yv <= h - 2)) v = 0.0f;
                    Vc = __float_as_int(v);
                    if (negKeys) Vc ^= (Vc >> 31) & 0x7fffffff;
                    Hc = max(Vc, lane_next(Vc));
                    Hc = max(Vc, lane_next(Hc));
                    hot = true;
                }
            }
        }

        // ---- Canny magnitude of this gradient row, as float bits (non-negative floats order like their
        //      bits), zero outside rows 1..h-2 and columns 1..w-1, column 0 below; u, v = at columns tx0-1+lane
        //      and tx0+lane
        int mag = __float_as_int(fabsf(gx) + fabsf(gy));
        if (!INNER) {
            const int xg = tx0 - 2 + lane;
            const bool rowOk = yg >= 1 && yg <= h - 2;
            if (!(rowOk && xg >= 1 && xg < w)) mag = 0;
            if (rowOk && tx0 == 0) {
                // CannySobel column 0 (ago_haf_cpu_canny.cpp:83-116 with the staged rows r0[-1] = 0 and
                // r1[-1] = r0[ALIGN16(w)-1]); luma lanes 3, 4 are x = 0, 1 and rows k-2..k are yg-1..yg+1.  It
                // is never an NMS centre, so its sector does not matter.
                const int a3 = __builtin_amdgcn_readlane((int)yC, 3), a4 = __builtin_amdgcn_readlane((int)yC, 4);
                const int b4 = __builtin_amdgcn_readlane((int)yD, 4);
                const int c3 = __builtin_amdgcn_readlane(yi, 3), c4 = __builtin_amdgcn_readlane(yi, 4);
                int t1_m1 = 0;
                if (w % 16 == 0) {
                    // column w-1 of a row is lane 2 (x = -1) of the row below it: rows k-1, k, and k+1, whose pixels
                    // are in pN
                    if (wide) {
                        t1_m1 = __builtin_amdgcn_readlane((int)yD, 2) + 2 * __builtin_amdgcn_readlane(yi, 2) +
                                __builtin_amdgcn_readlane(luma_of(k + 1, pN), 2);
                    } else {
                        t1_m1 = (int)yflat(F, P, yg - 1, w - 1) + (int)yflat(F, P, yg + 1, w - 1) + 2 * (int)yflat(F, P, yg, w - 1);
                    }
                }
                if (xg == 0) {
                    const int t0_1 = a4 + c4 + 2 * b4;
                    const int t1_0 = c3 - a3, t1_1 = c4 - a4;
                    mag = __float_as_int((float)(abs(t0_1) + abs(t1_m1 + 2 * t1_0 + t1_1)));
                }
            }
        }
        const int uk = lane_next(mag), vk = lane_next(uk);

        // ---- Canny NMS of tile row r = k-5 (image row ty0+r): rows uO/vO above, uN/vN the centre, uk/vk below; the
        //      larger of the two neighbours along the centre's sector (HafCpu_FastAtan2_Canny,
        //      ago_haf_cpu_arithmetic.cpp:9638-9656, on (gx, -gy): sector 1, or 3 where gx * -gy < 0; 0 where
        //      |gy| <= tan(22.5) |gx|; 2 where |gy| >= tan(67.5) |gx|, the last test wins)
        if (k >= 5 && k < TH + 5) {
            const int r = k - 5, y = ty0 + r;
            const int d0 = max(uN, lane_next(vN));      // left, right
            const int d1 = max(uk, lane_next(vO));      // lower left, upper right
            const int d2 = max(vO, vk);                 // above, below
            const int d3 = max(uO, lane_next(vk));      // upper left, lower right
            int nmax = in_mask(sec3 >> 2) ? d3 : d1;
            nmax = in_mask(sec0 >> 2) ? d0 : nmax;
            nmax = in_mask(sec2 >> 2) ? d2 : nmax;
            const uint64_t peak = mask_of(vN > nmax), up = mask_of(vN > P.upperBits), lo = mask_of(vN > P.lowerBits);
            const uint64_t valid = (INNER || (y >= 1 && y <= h - 2)) ? outCols : 0ull;
            const uint64_t sb = valid & ((peak & up) | P.upperAll);
            const uint64_t eb = valid & ((peak & (up | lo)) | P.upperAll | P.lowerAll);
            emLo = mvx_writelane((int)(uint32_t)eb, r, emLo);
            emHi = mvx_writelane((int)(uint32_t)(eb >> 32), r, emHi);
            smLo = mvx_writelane((int)(uint32_t)sb, r, smLo);
            smHi = mvx_writelane((int)(uint32_t)(sb >> 32), r, smHi);
        }
        {
            const float ax = fabsf(gx), ay = fabsf(gy);
            sec0 = mask_of(ay <= ax * 0.4142135623730950488016887242097f);
            sec2 = mask_of(ay >= ax * 2.4142135623730950488016887242097f);
            sec3 = mask_of((__float_as_int(gx) ^ __float_as_int(gy)) >= 0);   // (0 in either: sector 0 or 2)
        }

        // ---- Harris 3x3 NMS of tile row r = k-6: >= towards the upper-left half of the window, > towards the
        //      lower-right; without a score in the centre row there is no maximum
        if (k >= 6 && hotB) {
            const int r = k - 6, y = ty0 + r;
            // the lane shifts run with every lane active: a DPP read of a lane that a short-circuited
            // && has switched off returns 0, not that lane's value
            const int c = lane_next(Vb), cRight = lane_next(c);
            const uint64_t valid = (INNER || (y >= 1 && y <= h - 2)) ? outCols : 0ull;
            const uint64_t cb = valid & mask_of(c >= max(HO, Vb)) & mask_of(c > max(Hc, cRight));
            if (cb) {
                if (in_mask(cb)) {
                    const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(cb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)cb, 0u));
                    const uint32_t bits = negKeys ? (uint32_t)(c ^ ((c >> 31) & 0x7fffffff)) : (uint32_t)c;
                    cand[nc + below] = (uint64_t)(uint16_t)ox | ((uint64_t)(uint16_t)y << 16) | ((uint64_t)bits << 32);
                }
                nc += (uint32_t)__popcll(cb);
            }
        }
        // the new rows over the oldest ones
        yA = yk; dO = dk; sO = sk;
        xx0 = hxx; xy0 = hxy; yy0 = hyy;
        uO = uk; vO = vk; HO = Hc; Vb = Vc; hotB = hot;
    };

    uint32_t pf0 = 0, pf1 = 0;
    if (INNER || wide) { pf0 = fetch(0); pf1 = fetch(1); }
    float y0 = 0, y1 = 0, y2 = 0, y3 = 0, dA = 0, dB = 0, sA = 0, sB = 0;
    float xx0 = 0, xx1 = 0, xy0 = 0, xy1 = 0, yy0 = 0, yy1 = 0;
    int ua = 0, ub = 0, va = 0, vb = 0, Ha = 0, Hb = 0;
    static_assert(YH % 4 == 2, "four steps per loop trip, two after it");
    int k = 0;
    for (; k + 4 <= YH; k += 4) {
        step(k, pf0, pf1, y0, y1, y2, y3, dA, dB, sA, sB, xx0, xx1, xy0, xy1, yy0, yy1, ua, ub, va, vb, Ha, Hb);
        step(k + 1, pf1, pf0, y1, y2, y3, y0, dB, dA, sB, sA, xx1, xx0, xy1, xy0, yy1, yy0, ub, ua, vb, va, Hb, Ha);
        step(k + 2, pf0, pf1, y2, y3, y0, y1, dA, dB, sA, sB, xx0, xx1, xy0, xy1, yy0, yy1, ua, ub, va, vb, Ha, Hb);
        step(k + 3, pf1, pf0, y3, y0, y1, y2, dB, dA, sB, sA, xx1, xx0, xy1, xy0, yy1, yy0, ub, ua, vb, va, Hb, Ha);
    }
    step(k, pf0, pf1, y0, y1, y2, y3, dA, dB, sA, sB, xx0, xx1, xy0, xy1, yy0, yy1, ua, ub, va, vb, Ha, Hb);
    step(k + 1, pf1, pf0, y1, y2, y3, y0, dB, dA, sB, sA, xx1, xx0, xy1, xy0, yy1, yy0, ub, ua, vb, va, Hb, Ha);

    const __amdgpu_buffer_rsrc_t edR = plane_rsrc(F.edges);
    const uint32_t edStride = F.edgesStride;

    // ---- Harris candidates: one global atomic per tile, then the buffer copied out
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (nc) {
        uint32_t base = 0;
        if (lane == 0) base = __hip_atomic_fetch_add(gmem(F.candCount), nc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
        gptr_t<uint64_t> list = gmem((uint64_t *)F.cand);
        for (uint32_t i = (uint32_t)lane; i < nc; i += 64)
            if (base + i < P.candCap) list[base + i] = cand[i];
    }

    // ---- hysteresis inside the tile.  (a) Lanes 0..31 grow the edge pixels that a strong pixel reaches
    //      (the union of the 8-connected edge components holding a strong pixel), lanes 32..63 those a
    //      tile-border edge pixel reaches.  Edge pixels in neither are weak components inside the tile
    //      (-> 0); border-touching components without a strong pixel are undecided.
    static_assert(TH <= 32 && TW <= 63, "row masks: one lane per row in each half-wave");
    const int rr = lane & 31;
    const uint64_t emine = ((uint64_t)(uint32_t)emHi << 32) | (uint32_t)emLo, smine = ((uint64_t)(uint32_t)smHi << 32) | (uint32_t)smLo;
    const uint64_t e = __shfl(emine, rr);
    uint64_t seeds;
    if (lane < 32) seeds = __shfl(smine, rr);
    else seeds = (rr == 0 || rr == th - 1) ? e : (e & (1ull | (1ull << (tw - 1))));
    const uint64_t grown = grow_rows(seeds, e, lane);
    const uint64_t other = __shfl(grown, lane ^ 32);
    const uint64_t rm = lane < 32 ? grown : other;                  // lane r (both halves): reached from strong
    const uint64_t bmAll = lane < 32 ? (other & ~grown) : 0ull;     // lane r < 32: undecided

    //  (b) settle: reached -> 255; undecided -> 127 (k_resolve decides them); other edge pixels -> 0
    for (int r = 0; r < th; r++) {
        const uint64_t R = readlane64(rm, r), B = readlane64(bmAll, r);
        const int y = ty0 + r;
        const int v = in_mask(R) ? 255 : in_mask(B) ? 127 : 0;
        if (in_mask(outCols) && (INNER || (y >= 1 && y <= h - 2)))
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)v, edR, ox, (int)((uint32_t)y * edStride), 0);
    }

    //  (c) the undecided components, one at a time: the first set bit in row-major order is the
    //      component's smallest index p = row*TP + column; the k-th component found gets the id
    //      1 + tile*TNB + k (each touches a border pixel no other one does); flood it inside the
    //      undecided mask.  Border tables: top row, bottom row, left column, right column of the tile
    //      (actual extent): 0 for reached pixels (the strong node), the component id for undecided
    //      ones, -1 otherwise.
    int32_t topv = -1, botv = -1, leftv = -1, rightv = -1;
    {
        const uint64_t R0 = readlane64(rm, 0), Rb = readlane64(rm, th - 1);
        topv = in_mask(R0) ? 0 : topv;     // the masks hold no column past the tile's width
        botv = in_mask(Rb) ? 0 : botv;
        if (lane < th && (rm & 1ull)) leftv = 0;
        if (lane < th && ((rm >> (tw - 1)) & 1ull)) rightv = 0;
    }
    gptr_t<uint32_t> ulist = gmem(F.ulist) + (size_t)tile * TS;
    uint32_t nU = 0, nComp = 0;
    uint64_t bm = bmAll;
    while (true) {
        const uint64_t rows = __ballot(bm != 0ull);
        if (!rows) break;
        const int r0 = __builtin_ctzll(rows);
        const int c0 = __builtin_ctzll(readlane64(bm, r0));
        const uint32_t gid = 1u + (uint32_t)tile * TNB + nComp;
        const uint64_t c = grow_rows(lane == r0 ? (1ull << c0) : 0ull, bm, lane);
        if (lane == 0) gmem(F.parent)[gid] = gid;
        const uint64_t C0 = readlane64(c, 0), Cb = readlane64(c, th - 1);
        topv = in_mask(C0) ? (int32_t)gid : topv;
        botv = in_mask(Cb) ? (int32_t)gid : botv;
        if (lane < th && (c & 1ull)) leftv = (int32_t)gid;
        if (lane < th && ((c >> (tw - 1)) & 1ull)) rightv = (int32_t)gid;
        // list the component's pixels for k_resolve: p | k << 16
        uint64_t crow = __ballot(c != 0ull);
        while (crow) {
            const int r = __builtin_ctzll(crow);
            crow &= crow - 1;
            const uint64_t m = readlane64(c, r);
            if (in_mask(m)) {
                const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                ulist[nU + below] = (uint32_t)(r * TP + lane) | (nComp << 16);
            }
            nU += (uint32_t)__popcll(m);
        }
        bm &= ~c;
        nComp++;
    }
    gptr_t<int32_t> bt = gmem(F.border) + (long)tile * 2 * (TW + TH);
    if (lane < TW) { bt[lane] = topv; bt[TW + lane] = botv; }
    if (lane < TH) { bt[2 * TW + lane] = leftv; bt[2 * TW + TH + lane] = rightv; }
    if (lane == 0) gmem(F.ucount)[tile] = nU;
}

__global__ void __launch_bounds__(64 * FTW)
k_front(const FrameDesc *__restrict__ frames, GraphParams P)
{
    __shared__ uint64_t candLds[FTW][CAND_MAX];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int tX = (int)blockIdx.x * FTW + wave, tY = (int)blockIdx.y;
    if (tX >= P.tilesX) return;
    const int tile = tY * P.tilesX + tX;
    const int tx0 = tX * TW, ty0 = tY * TH;
    const bool inner = tx0 >= 4 && tx0 + TW + 4 <= P.w && ty0 >= 4 && ty0 + TH + 4 <= P.h;
    const FrameDesc &F = frames[blockIdx.z];   // fields are read where they are used: the stream needs the scalar registers
    if (inner) front_tile<true>(candLds[wave], F, P, tx0, ty0, tile);
    else front_tile<false>(candLds[wave], F, P, tx0, ty0, tile);
}

// union the border components of each tile with those of its right, lower and diagonal neighbours;
// one wave per tile (lane = row of the right column, then column of the bottom row), four tiles per
// workgroup
__global__ void __launch_bounds__(256)
k_border(const FrameDesc *__restrict__ frames, GraphParams P)
{
    static_assert(TW <= 64 && TH <= 64, "one lane per border pixel");
    const FrameDesc &F = frames[blockIdx.z];
    const int lane = (int)threadIdx.x & 63;
    const int tile = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (tile >= P.tilesX * P.tilesY) return;
    const int tX = tile % P.tilesX, tYi = tile / P.tilesX;
    const int tw = min(TW, P.w - tX * TW), th = min(TH, P.h - tYi * TH);
    gptr_t<const int32_t> tables = gmem((const int32_t *)F.border);
    gptr_t<const int32_t> bt = tables + (long)tile * 2 * (TW + TH);
    gptr_t<uint32_t> par = gmem(F.parent);
    // all table reads first, so that the wave waits for memory once: my right column (rows 0..th-1) and its
    // right neighbour's left column, |dr| <= 1; my bottom row and the top row below it (the tile below has the
    // same width), |dc| <= 1; the corners of the lower right and lower left tiles (the latter of full width)
    const bool right = tX + 1 < P.tilesX, down = tYi + 1 < P.tilesY;
    gptr_t<const int32_t> nr = tables + (long)(tile + 1) * 2 * (TW + TH), nd = tables + (long)(tile + P.tilesX) * 2 * (TW + TH);
    const int32_t ra = right && lane < th ? bt[2 * TW + TH + lane] : -1, rb = right && lane < th ? nr[2 * TW + lane] : -1;
    const int32_t da = down && lane < tw ? bt[TW + lane] : -1, db = down && lane < tw ? nd[lane] : -1;
    const int32_t cr = down && right ? (nd + 2 * (TW + TH))[0] : -1, cl = down && tX > 0 ? (nd - 2 * (TW + TH))[TW - 1] : -1;
    const int32_t ar = __builtin_amdgcn_readlane(da, tw - 1), al = __builtin_amdgcn_readlane(da, 0);
    border_unions(par, ra, rb, lane);
    border_unions(par, da, db, lane);
    if (lane == 0 && ar >= 0 && cr >= 0) gunion(par, (uint32_t)ar, (uint32_t)cr);
    if (lane == 0 && al >= 0 && cl >= 0) gunion(par, (uint32_t)al, (uint32_t)cl);
}

// the undecided pixels k_front listed take the state of their component's global root (strong iff
// the root is node 0); one wave per tile, four tiles per workgroup
__global__ void __launch_bounds__(256)
k_resolve(const FrameDesc *__restrict__ frames, GraphParams P)
{
    const FrameDesc &F = frames[blockIdx.z];
    const int lane = (int)threadIdx.x & 63;
    const int w0 = ((int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * RES_TILES;
    const int tiles = P.tilesX * P.tilesY;
    if (w0 >= tiles) return;
    // the wave's tiles side by side: their counts, the first 64 entries of their lists (whatever the list
    // holds past its count is not used) and then the roots of all of them, so that a wave waits for memory
    // about three times however many of its tiles list pixels
    const uint32_t cnt = (lane < RES_TILES && w0 + lane < tiles) ? gmem(F.ucount)[w0 + lane] : 0u;
    uint32_t e[RES_TILES];
#pragma unroll
    for (int j = 0; j < RES_TILES; j++) e[j] = w0 + j < tiles ? gmem((const uint32_t *)F.ulist)[(size_t)(w0 + j) * TS + lane] : 0u;
    if (!__any(cnt != 0u)) return;
    gptr_t<uint32_t> par = gmem(F.parent);
    gptr_t<uint8_t> edges = gmem(F.edges);
    const auto put = [&](int tile, uint32_t entry, uint32_t root) {
        const uint32_t p = entry & 0xffffu;
        edges[(long)((tile / P.tilesX) * TH + (int)(p / TP)) * F.edgesStride + (tile % P.tilesX) * TW + (int)(p % TP)] = (root == 0) ? 255 : 0;
    };
    uint32_t g[RES_TILES], up[RES_TILES];
    bool has[RES_TILES];
#pragma unroll
    for (int j = 0; j < RES_TILES; j++) {
        has[j] = lane < __builtin_amdgcn_readlane((int)cnt, j);
        g[j] = has[j] ? 1u + (uint32_t)(w0 + j) * TNB + (e[j] >> 16) : 0u;
        up[j] = has[j] ? par[g[j]] : 0u;
    }
    // most chains are a few links, and the cached loads are the shortest for those; from the fifth link on they are
    // shortened as they are walked, by loads past the L1, which would hide what other compute units have shortened
    // (serpentines of 12-column steps through 3840x2160: 154 us with plain finds, 115 with cached loads, 63 so)
    for (int n = 0;; n++) {
        bool more = false;
#pragma unroll
        for (int j = 0; j < RES_TILES; j++) {
            if (up[j] != g[j]) {
                const uint32_t l = up[j];
                up[j] = n < 4 ? par[l] : gstep<__HIP_MEMORY_SCOPE_AGENT>(par, g[j], l);
                g[j] = l;
                more = true;
            }
        }
        if (!__any(more)) break;
    }
#pragma unroll
    for (int j = 0; j < RES_TILES; j++) {
        if (has[j]) put(w0 + j, e[j], g[j]);
        for (uint32_t i = 64u + (uint32_t)lane; i < (uint32_t)__builtin_amdgcn_readlane((int)cnt, j); i += 64) {
            const uint32_t entry = gmem((const uint32_t *)F.ulist)[(size_t)(w0 + j) * TS + i];
            put(w0 + j, entry, gfind_settled<__HIP_MEMORY_SCOPE_AGENT>(par, 1u + (uint32_t)(w0 + j) * TNB + (entry >> 16)));
        }
    }
}

// pyramid level `lvl` (>= 2) from level lvl-1, all frames
__global__ void __launch_bounds__(256)
k_half_batched(const FrameDesc *__restrict__ frames, GraphParams P, int lvl)
{
    const FrameDesc &F = frames[blockIdx.z];
    const int y = 1 + (int)(blockIdx.y * 4) + __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    if (y <= P.lvlH[lvl] - 2)
        half_row((uint32_t)P.lvlW[lvl], F.lvl[lvl], F.lvlStride[lvl], (uint32_t)P.lvlW[lvl - 1], (uint32_t)P.lvlH[lvl - 1],
                 F.lvl[lvl - 1], F.lvlStride[lvl - 1], blockIdx.x * PYR_CHUNKS, y);
}

// Harris sort and pick, one workgroup per frame; clears the candidate count for the next batch
__global__ void __launch_bounds__(PICK_THREADS)
k_pick_batched(const FrameDesc *__restrict__ frames, GraphParams P)
{
    const FrameDesc &F = frames[blockIdx.x];
    const PickWork W = *reinterpret_cast<const PickWork *>(F.pickWs);
    harris_pick_block((const XYS *)F.cand, F.candCount, true, P.candCap, P.dist, (uint32_t)P.w, (uint32_t)P.h,
                      (Keypoint *)F.corners, P.capacity, F.numItems, F.count, W);
}

__global__ void k_fill_bytes(uint32_t *p, uint32_t v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// ---------------------------------------------------------------- host side -----------------------
struct GraphLayout {
    size_t descs, frameBytes, border, parent, ulist, ucount, cand, candCount, pickHdr, pickWs, total;
    uint32_t tiles, candCap;
};

inline GraphLayout graph_layout(const mvx_vision_params_t &p, uint32_t maxFrames)
{
    GraphLayout L;
    const uint32_t tx = (p.width + TW - 1) / TW, ty = (p.height + TH - 1) / TH;
    L.tiles = tx * ty;
    L.candCap = std::max(1u, ((p.width - 1) / 2) * ((p.height - 1) / 2));   // NMS maxima are never 8-adjacent
    L.descs = align256(sizeof(FrameDesc) * (size_t)maxFrames);
    size_t o = 0;
    L.border = o;    o = align256(o + (size_t)L.tiles * 2 * (TW + TH) * 4);
    L.parent = o;    o = align256(o + ((size_t)L.tiles * TNB + 1) * 4);
    L.ulist = o;     o = align256(o + (size_t)L.tiles * TS * 4);
    L.ucount = o;    o = align256(o + (size_t)L.tiles * 4);
    L.cand = o;      o = align256(o + (size_t)L.candCap * sizeof(XYS));
    L.candCount = o; o = align256(o + 4);
    L.pickHdr = o;   o = align256(o + sizeof(PickWork));
    L.pickWs = o;    o = align256(o + pick_layout(L.candCap).total);
    L.frameBytes = o;
    L.total = L.descs + L.frameBytes * maxFrames;
    return L;
}

inline bool params_ok(const mvx_vision_params_t &p)
{
    if (!(p.width >= 16 && p.height >= 16 && (p.width % 4) == 0 && p.width <= 32767 && p.height <= 32767 &&
          (p.height % 2) == 0 && p.scaledWidth == p.width / 2 && p.scaledHeight == p.height / 2 && p.levels >= 1 &&
          p.levels <= 8 && p.harrisMinDistance > 0.0f))
        return false;
    // every pyramid step must be one the reference accepts (source >= 5, destination >= 3)
    uint32_t lw = p.width, lh = p.height;
    for (uint32_t l = 1; l < p.levels; l++) {
        const uint32_t nw = (lw + 1) / 2, nh = (lh + 1) / 2;
        if (lw < 5 || lh < 5 || nw < 3 || nh < 3) return false;
        lw = nw; lh = nh;
    }
    return true;
}

inline GraphParams graph_params(const mvx_vision_params_t &p, const GraphLayout &L)
{
    GraphParams P;
    P.w = (int)p.width; P.h = (int)p.height;
    P.yStride = (int)((p.width + 15) & ~15u);
    P.tilesX = (int)((p.width + TW - 1) / TW); P.tilesY = (int)((p.height + TH - 1) / TH);
    P.dw = (int)p.scaledWidth; P.dh = (int)p.scaledHeight;
    P.levels = (int)p.levels;
    uint32_t lw = p.width, lh = p.height;
    for (int l = 0; l < 8; l++) { P.lvlW[l] = (int)lw; P.lvlH[l] = (int)lh; lw = (lw + 1) / 2; lh = (lh + 1) / 2; }
    P.lower = p.cannyLower; P.upper = p.cannyUpper;
    P.k = p.harrisK; P.thr = p.harrisThreshold; P.dist = p.harrisMinDistance;
    // normFactor of ago_kernel_api.cpp:16941-16942 for gradient size 3, in float, left to right
    float nf = 255.0f * (float)(1 << 2) * 3;
    P.norm = nf * nf * nf * nf;
    P.normRcp = recip_rn(P.norm);
    // RN(mc / norm) > thr implies mc > thr * norm; the product is exact in double and rounds down here, and
    // mc <= RN(gx2 * gy2) when k >= 0.  Negative (or NaN) thr and k: every row takes the full path.
    P.hotMc = P.hotProd = -INFINITY;
    if (P.thr >= 0.0f) {
        const double m = (double)P.thr * (double)P.norm;
        float f = (float)m;
        if ((double)f > m) f = std::nextafter(f, 0.0f);
        P.hotMc = f;
        if (P.k >= 0.0f) P.hotProd = f;
    }
    const auto bits = [](uint32_t t) { const float f = (float)std::max((int)t, 0); int b; memcpy(&b, &f, 4); return b; };
    P.upperBits = bits(P.upper); P.lowerBits = bits(P.lower);
    P.upperAll = (int)P.upper < 0 ? ~0ull : 0ull;
    P.lowerAll = (int)P.lower < 0 ? ~0ull : 0ull;
    P.capacity = p.cornerCapacity;
    P.candCap = L.candCap;
    return P;
}

inline bool plane_ok_v(const void *ptr, uint32_t w, uint32_t stride, uint32_t bpp)
{
    return ptr && aligned16(ptr) && (stride % 16u) == 0 && stride >= ((w * bpp + 15u) & ~15u);
}

}  // namespace mvx

using namespace mvx;

extern "C" int mvx_VisionGraph_supported(const mvx_vision_params_t *p) { return (p && params_ok(*p)) ? 1 : 0; }

extern "C" size_t mvx_VisionGraph_workspace_size(const mvx_vision_params_t *p, uint32_t maxFrames)
{
    if (!p || !params_ok(*p) || maxFrames == 0) return 0;
    return graph_layout(*p, maxFrames).total;
}

extern "C" int mvx_VisionGraph_prepare(mvx_stream_t stream, const mvx_vision_params_t *p, const mvx_vision_frame_t *frames,
                                       uint32_t nframes, void *workspace, size_t workspaceSize)
{
    if (!p || !params_ok(*p) || !frames || nframes == 0 || !workspace) return MVX_ERROR_INVALID_PARAMETERS;
    const GraphLayout L = graph_layout(*p, nframes);
    if (workspaceSize < L.total || !aligned16(workspace)) return MVX_ERROR_INVALID_PARAMETERS;
    std::vector<FrameDesc> D(nframes);
    uint8_t *base = (uint8_t *)workspace + L.descs;
    uint32_t lw = p->width, lh = p->height;
    for (uint32_t f = 0; f < nframes; f++) {
        const mvx_vision_frame_t &in = frames[f];
        FrameDesc &d = D[f];
        memset(&d, 0, sizeof(d));
        if (!plane_ok_v(in.rgb, p->width, in.rgbStride, 3) || !plane_ok_v(in.scaled, p->scaledWidth, in.scaledStride, 1) ||
            !plane_ok_v(in.edges, p->width, in.edgesStride, 1) || !in.corners || !in.numItems || !in.numCorners)
            return MVX_ERROR_INVALID_PARAMETERS;
        lw = p->width; lh = p->height;
        for (uint32_t l = 0; l < p->levels; l++) {
            if (!plane_ok_v(in.pyramid[l], lw, in.pyramidStride[l], 1)) return MVX_ERROR_INVALID_PARAMETERS;
            d.lvl[l] = in.pyramid[l];
            d.lvlStride[l] = in.pyramidStride[l];
            lw = (lw + 1) / 2; lh = (lh + 1) / 2;
        }
        d.rgb = in.rgb; d.rgbStride = in.rgbStride;
        d.scaled = in.scaled; d.scaledStride = in.scaledStride;
        d.edges = in.edges; d.edgesStride = in.edgesStride;
        d.corners = in.corners; d.numItems = in.numItems; d.count = in.numCorners;
        uint8_t *fb = base + (size_t)f * L.frameBytes;
        d.border = (int32_t *)(fb + L.border);
        d.parent = (uint32_t *)(fb + L.parent);
        d.ulist = (uint32_t *)(fb + L.ulist);
        d.ucount = (uint32_t *)(fb + L.ucount);
        d.cand = fb + L.cand;
        d.candCount = (uint32_t *)(fb + L.candCount);
        d.pickWs = fb + L.pickHdr;
        // the pick workspace header holds the device pointers of the frame's pick scratch
        const PickWork W = pick_work(fb + L.pickWs, L.candCap);
        if (hipMemcpy(fb + L.pickHdr, &W, sizeof(W), hipMemcpyHostToDevice) != hipSuccess) return MVX_FAILURE;
        const PickLayout PL = pick_layout(L.candCap);
        hipLaunchKernelGGL(k_fill_bytes, dim3(256), dim3(256), 0, stream_of(stream), (uint32_t *)(fb + L.pickWs + PL.hkey),
                           HASH_EMPTY, (size_t)PL.hsize);
        hipLaunchKernelGGL(k_fill_bytes, dim3(1), dim3(64), 0, stream_of(stream), d.candCount, 0u, (size_t)1);
        // union-find slot 0 is the strong node every strong tile-border pixel maps to: its own root
        hipLaunchKernelGGL(k_fill_bytes, dim3(1), dim3(64), 0, stream_of(stream), d.parent, 0u, (size_t)1);
    }
    if (hipMemcpy(workspace, D.data(), sizeof(FrameDesc) * nframes, hipMemcpyHostToDevice) != hipSuccess) return MVX_FAILURE;
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

namespace mvx {

// one stage for the frames D[0 .. nframes-1]
static void launch_stage(hipStream_t s, const GraphParams &P, const FrameDesc *D, uint32_t nframes, int stage)
{
    switch (stage) {
    case 0:
        hipLaunchKernelGGL(k_front, dim3((P.tilesX + FTW - 1) / FTW, P.tilesY, nframes), dim3(64 * FTW), 0, s, D, P);
        break;
    case 1:
        hipLaunchKernelGGL(k_border, dim3((P.tilesX * P.tilesY + 3) / 4, 1, nframes), dim3(256), 0, s, D, P);
        break;
    case 2:
        hipLaunchKernelGGL(k_resolve, dim3((P.tilesX * P.tilesY + 4 * RES_TILES - 1) / (4 * RES_TILES), 1, nframes), dim3(256), 0,
                           s, D, P);
        break;
    case 3:
        for (int l = 2; l < P.levels; l++)
            hipLaunchKernelGGL(k_half_batched, half_grid((uint32_t)P.lvlW[l], (uint32_t)P.lvlH[l], nframes), dim3(64, 4), 0, s, D, P, l);
        break;
    case 4:
        hipLaunchKernelGGL(k_pick_batched, dim3(nframes), dim3(PICK_THREADS), 0, s, D, P);
        break;
    }
}

}  // namespace mvx

extern "C" int mvx_VisionGraph_run_stage_range(mvx_stream_t stream, const mvx_vision_params_t *p, uint32_t firstFrame,
                                               uint32_t nframes, void *workspace, size_t workspaceSize, int stage)
{
    if (!p || !params_ok(*p) || nframes == 0 || !workspace || stage < 0 || stage >= MVX_VISION_STAGES ||
        firstFrame > UINT32_MAX - nframes)
        return MVX_ERROR_INVALID_PARAMETERS;
    const GraphLayout L = graph_layout(*p, firstFrame + nframes);
    if (workspaceSize < L.total) return MVX_ERROR_INVALID_PARAMETERS;
    launch_stage(stream_of(stream), graph_params(*p, L), (const FrameDesc *)workspace + firstFrame, nframes, stage);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" int mvx_VisionGraph_run_stage(mvx_stream_t stream, const mvx_vision_params_t *p, uint32_t nframes,
                                         void *workspace, size_t workspaceSize, int stage)
{
    return mvx_VisionGraph_run_stage_range(stream, p, 0, nframes, workspace, workspaceSize, stage);
}

// A lane: the streams the per-frame stages after the fused tile pass run on -- one for the two
// hysteresis stages, one for the pyramid levels 2.. and the Harris pick -- with the fork and join
// events, all at the default priority.  Each engine graph owns one (mvx_VisionGraph_lane_create at
// verification, destroyed with the graph), so concurrent graphs never share a side stream;
// mvx_VisionGraph_run uses one shared lane per device, created on first use and kept until the
// process ends, whose mutex orders the callers that share it.
struct mvx_vision_lane {
    hipStream_t stream = nullptr, hyst = nullptr;
    hipEvent_t fork = nullptr, join = nullptr, joinHyst = nullptr;
    std::mutex mu;
};

namespace mvx {

static int lane_init(mvx_vision_lane *L)
{
    if (hipStreamCreateWithFlags(&L->stream, hipStreamNonBlocking) != hipSuccess) return MVX_FAILURE;
    if (hipStreamCreateWithFlags(&L->hyst, hipStreamNonBlocking) != hipSuccess) return MVX_FAILURE;
    if (hipEventCreateWithFlags(&L->fork, hipEventDisableTiming) != hipSuccess) return MVX_FAILURE;
    if (hipEventCreateWithFlags(&L->join, hipEventDisableTiming) != hipSuccess) return MVX_FAILURE;
    if (hipEventCreateWithFlags(&L->joinHyst, hipEventDisableTiming) != hipSuccess) return MVX_FAILURE;
    return MVX_SUCCESS;
}

// frames per chunk of the pipelined run: by default all frames in one chunk.  Smaller chunks overlap a
// chunk's later stages with the next chunk's tile pass, but measured slower on MI355X (16 frames in one chunk,
// in two, in four: 540, 569 and 633 us at 3840x2160, 183, 221 and 276 at 1920x1080, 124, 150 and 231 at
// 1284x726): the tile pass is bound by VALU issue, and the latency-bound union-find and pick waves resident
// beside it slow it by more than they hide.
static uint32_t mvx_vision_default_chunk(uint32_t nframes) { return nframes; }

static void lane_free(mvx_vision_lane *L)
{
    if (L->joinHyst) (void)hipEventDestroy(L->joinHyst);
    if (L->join) (void)hipEventDestroy(L->join);
    if (L->fork) (void)hipEventDestroy(L->fork);
    if (L->hyst) (void)hipStreamDestroy(L->hyst);
    if (L->stream) (void)hipStreamDestroy(L->stream);
    L->joinHyst = L->join = L->fork = nullptr;
    L->hyst = L->stream = nullptr;
}

static std::mutex g_sharedMu;
static mvx_vision_lane *g_shared[64];
static bool g_sharedTried[64];

static mvx_vision_lane *shared_lane()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> lk(g_sharedMu);
    if (!g_sharedTried[dev]) {
        g_sharedTried[dev] = true;
        mvx_vision_lane *L = new mvx_vision_lane();
        if (lane_init(L) == MVX_SUCCESS) g_shared[dev] = L;
        else { lane_free(L); delete L; }
    }
    return g_shared[dev];
}

}  // namespace mvx

extern "C" int mvx_VisionGraph_lane_create(mvx_vision_lane_t **lane)
{
    if (!lane) return MVX_ERROR_INVALID_PARAMETERS;
    *lane = nullptr;
    mvx_vision_lane *L = new mvx_vision_lane();
    const int rc = lane_init(L);
    if (rc) { lane_free(L); delete L; return rc; }
    *lane = L;
    return MVX_SUCCESS;
}

extern "C" int mvx_VisionGraph_lane_destroy(mvx_vision_lane_t *lane)
{
    if (!lane) return MVX_SUCCESS;
    (void)hipStreamSynchronize(lane->stream);
    (void)hipStreamSynchronize(lane->hyst);
    lane_free(lane);
    delete lane;
    return MVX_SUCCESS;
}

// The frames go through in chunks of framesPerChunk: the fused tile pass of each chunk on the caller's
// stream, then -- once it has finished, while the caller's stream goes on with the next chunk's tile
// pass -- that chunk's hysteresis stages on one lane stream and its pyramid levels and Harris pick on the
// other (the last chunk's hysteresis on the caller's stream and its pick on the first).  At the end the caller's stream waits for both
// lane streams, so the call orders like a single-stream sequence.  Fork and join are event waits, which a hipGraph capture of the caller's
// stream records as dependencies.  Once forked, the joins are recorded and waited for on every path,
// errors included, so a captured caller stream is never left forked.
extern "C" int mvx_VisionGraph_run_pipelined(mvx_stream_t stream, mvx_vision_lane_t *lane, const mvx_vision_params_t *p,
                                             uint32_t nframes, void *workspace, size_t workspaceSize,
                                             uint32_t framesPerChunk)
{
    if (!p || !params_ok(*p) || nframes == 0 || !workspace) return MVX_ERROR_INVALID_PARAMETERS;
    const GraphLayout L = graph_layout(*p, nframes);
    if (workspaceSize < L.total) return MVX_ERROR_INVALID_PARAMETERS;
    const GraphParams P = graph_params(*p, L);
    const FrameDesc *D = (const FrameDesc *)workspace;
    hipStream_t main = stream_of(stream);
    if (!lane) {
        for (int st = 0; st < MVX_VISION_STAGES; st++) launch_stage(main, P, D, nframes, st);
        MVX_LAUNCH_CHECK();
        return MVX_SUCCESS;
    }
    const uint32_t chunk = framesPerChunk ? std::min(framesPerChunk, nframes) : mvx_vision_default_chunk(nframes);
    std::lock_guard<std::mutex> lock(lane->mu);
    int rc = MVX_SUCCESS;
    bool forked = false;
    for (uint32_t f0 = 0; f0 < nframes && !rc; f0 += chunk) {
        const uint32_t n = std::min(chunk, nframes - f0);
        launch_stage(main, P, D + f0, n, 0);
        if (hipEventRecord(lane->fork, main) != hipSuccess || hipStreamWaitEvent(lane->hyst, lane->fork, 0) != hipSuccess ||
            hipStreamWaitEvent(lane->stream, lane->fork, 0) != hipSuccess) {
            rc = MVX_FAILURE;
            break;
        }
        forked = true;
        // the last chunk's hysteresis follows its tile pass on the caller's stream: no stream hop on
        // the critical path; its Harris pick then has the other lane stream to itself
        const bool last = f0 + n >= nframes;
        hipStream_t hs = last ? main : lane->hyst;
        launch_stage(last ? lane->hyst : lane->stream, P, D + f0, n, 4);
        launch_stage(lane->stream, P, D + f0, n, 3);
        launch_stage(hs, P, D + f0, n, 1);
        launch_stage(hs, P, D + f0, n, 2);
        if (hipGetLastError() != hipSuccess) rc = MVX_ERROR_LAUNCH;
    }
    if (forked) {
        const bool j1 = hipEventRecord(lane->joinHyst, lane->hyst) == hipSuccess &&
                        hipStreamWaitEvent(main, lane->joinHyst, 0) == hipSuccess;
        const bool j2 = hipEventRecord(lane->join, lane->stream) == hipSuccess &&
                        hipStreamWaitEvent(main, lane->join, 0) == hipSuccess;
        if (!rc && !(j1 && j2)) rc = MVX_FAILURE;
    }
    return rc;
}

extern "C" int mvx_VisionGraph_run_lane(mvx_stream_t stream, mvx_vision_lane_t *lane, const mvx_vision_params_t *p,
                                        uint32_t nframes, void *workspace, size_t workspaceSize)
{
    return mvx_VisionGraph_run_pipelined(stream, lane, p, nframes, workspace, workspaceSize, 0);
}

extern "C" int mvx_VisionGraph_run(mvx_stream_t stream, const mvx_vision_params_t *p, uint32_t nframes, void *workspace,
                                   size_t workspaceSize)
{
    return mvx_VisionGraph_run_lane(stream, shared_lane(), p, nframes, workspace, workspaceSize);
}
