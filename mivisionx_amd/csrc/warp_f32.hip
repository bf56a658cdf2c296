// warp_f32.hip -- differentiable F32 bilinear WarpPerspective and Remap, their adjoints, a fused
// L2 photometric loss with its gradient, and the F32 half-scale Gaussian pyramid with its adjoint.
//
// The reference has no F32 warp and no adjoint (its warps are U8, ago_haf_cpu_geometric.cpp:1579
// and :249); this is the differentiable counterpart used for gradient-based image alignment.  The
// sampling convention is the reference's: a destination pixel (x, y) samples the source at
// (u, v) = ((h0 x + h1 y + h2) / z, (h3 x + h4 y + h5) / z), z = h6 x + h7 y + h8 (the OpenVX matrix
// maps destination to source), bilinearly from the four pixels around (u, v); source pixels
// outside [0, sw) x [0, sh) read 0 (constant border 0), and a destination pixel with z <= 0 or a
// non-finite sample position is 0 with zero gradient.  Zero padding keeps the warp continuous in
// (u, v) everywhere, so its adjoint is the derivative almost everywhere.
//
// Adjoints, for g = dL/d out(x, y):
//   dL/d src   scatter-add of g times the four bilinear weights (hardware F32 atomics; the order of
//              additions is not fixed, so the last bit may vary between runs);
//   dL/d H     Iu = (1-fy)(p01-p00) + fy(p11-p10), Iv = (1-fx)(p10-p00) + fx(p11-p01),
//              a = g Iu / z, b = g Iv / z, c = -(a u + b v):
//              dH = (a x, a y, a, b x, b y, b, c x, c y, c), summed over the image -- per workgroup
//              in F32, then across workgroups in F64 by a second kernel in a fixed order, so dH
//              is deterministic.
//   dL/d map   (Remap) per pixel (g Iu, g Iv).
// Images of one call share a size; `count` images lie at a fixed byte distance (batch stride).
#include "mvx_common.hpp"
#include <climits>
#include <type_traits>

namespace mvx {

constexpr int WF_BX = 64, WF_BY = 4, WF_ROWS = 4;   // block 64x4 threads, each 4 rows: 64x16 px
constexpr int WF_TILE_W = WF_BX, WF_TILE_H = WF_BY * WF_ROWS;
constexpr int WF_SLOTS = 10;                        // 9 dH entries + loss

struct F32Plane {
    const float *p;
    uint32_t w, h, stride;  // stride in bytes
    size_t batch;           // bytes between images
};

MVX_DEV const float *row_of(const F32Plane &P, uint32_t img, int y)
{
    return (const float *)((const uint8_t *)P.p + img * P.batch + (size_t)y * P.stride);
}

MVX_DEV float px(const F32Plane &P, uint32_t img, int x, int y)
{
    return (x >= 0 && y >= 0 && x < (int)P.w && y < (int)P.h) ? row_of(P, img, y)[x] : 0.f;
}

// two neighbouring pixels at any 4-byte aligned address
struct __attribute__((packed, aligned(4))) float2a {
    float x, y;
};

// one bilinear sample with everything the adjoint needs
struct Sample {
    bool ok;
    int x0, y0;
    float fx, fy, p00, p01, p10, p11, val;
};

// sample at (bx + du, by + dv) for integers bx, by: the split into cell and fraction is taken on
// the offsets, so the fraction keeps the precision of |du| rather than of |bx + du|
MVX_DEV Sample bilinear(const F32Plane &S, uint32_t img, int bx, int by, float du, float dv)
{
    Sample s;
    s.ok = fabsf(du) < 1.0e7f && fabsf(dv) < 1.0e7f;   // also false for NaN
    if (!s.ok) { s.val = 0.f; return s; }
    const float fu = floorf(du), fv = floorf(dv);
    s.x0 = bx + (int)fu; s.y0 = by + (int)fv;
    s.fx = du - fu; s.fy = dv - fv;
    s.p00 = px(S, img, s.x0, s.y0);     s.p01 = px(S, img, s.x0 + 1, s.y0);
    s.p10 = px(S, img, s.x0, s.y0 + 1); s.p11 = px(S, img, s.x0 + 1, s.y0 + 1);
    s.val = (1.f - s.fy) * ((1.f - s.fx) * s.p00 + s.fx * s.p01) + s.fy * ((1.f - s.fx) * s.p10 + s.fx * s.p11);
    return s;
}

MVX_DEV void scatter(float *gsrc, uint32_t gStride, uint32_t w, uint32_t h, const Sample &s, float g)
{
    const float wts[4] = {(1.f - s.fx) * (1.f - s.fy), s.fx * (1.f - s.fy), (1.f - s.fx) * s.fy, s.fx * s.fy};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int x = s.x0 + (k & 1), y = s.y0 + (k >> 1);
        if (x >= 0 && y >= 0 && x < (int)w && y < (int)h && wts[k] != 0.f)
            atomicAdd((float *)((uint8_t *)gsrc + (size_t)y * gStride) + x, g * wts[k]);
    }
}

// The homography arrives in F64 and is used in F32 as {h0 - h8, h1, h2, h3, h4 - h8, h5, h6, h7, h8}:
// the two differences are formed in F64, so a near-identity matrix loses nothing when it is rounded
// (rounding h0 and h8 separately would shift the sample by ~1e-7 x its coordinate).
struct HomF {
    float d0, h1, h2, h3, d4, h5, h6, h7, h8;
};

MVX_DEV HomF load_hom(const double *H)
{
    HomF m;
    m.d0 = (float)(H[0] - H[8]); m.h1 = (float)H[1]; m.h2 = (float)H[2];
    m.h3 = (float)H[3]; m.d4 = (float)(H[4] - H[8]); m.h5 = (float)H[5];
    m.h6 = (float)H[6]; m.h7 = (float)H[7]; m.h8 = (float)H[8];
    return m;
}

// sample position of destination pixel (X, Y) as offsets from it: du = u - X = (h0 X + h1 Y + h2 -
// X z) / z, regrouped as ((h0 - h8) X + h1 Y + h2 - X (h6 X + h7 Y)) / z (and likewise dv), which
// for near-identity homographies is far better conditioned in F32 than u itself
MVX_DEV bool project(const HomF &H, float X, float Y, float &du, float &dv, float &z)
{
    const float q = H.h6 * X + H.h7 * Y;
    z = q + H.h8;
    if (!(z > 0.f)) return false;
    du = ((H.d0 * X + H.h1 * Y + H.h2) - X * q) / z;
    dv = ((H.h3 * X + H.d4 * Y + H.h5) - Y * q) / z;
    return true;
}

// ------------------------------------------------------------------ forward kernels --------------
__global__ void __launch_bounds__(WF_BX * WF_BY)
k_warp_f32(F32Plane S, float *dst, uint32_t dw, uint32_t dh, uint32_t dStride, size_t dBatch, const double *Hs)
{
    const uint32_t img = blockIdx.z;
    const int x = blockIdx.x * WF_BX + threadIdx.x;
    const HomF H = load_hom(Hs + 9 * img);
    for (int r = 0; r < WF_ROWS; r++) {
        const int y = blockIdx.y * WF_TILE_H + r * WF_BY + threadIdx.y;
        if (x >= (int)dw || y >= (int)dh) continue;
        float du, dv, z, out = 0.f;
        if (project(H, (float)x, (float)y, du, dv, z)) out = bilinear(S, img, x, y, du, dv).val;
        ((float *)((uint8_t *)dst + img * dBatch + (size_t)y * dStride))[x] = out;
    }
}

__global__ void __launch_bounds__(WF_BX * WF_BY)
k_remap_f32(F32Plane S, float *dst, uint32_t dw, uint32_t dh, uint32_t dStride, size_t dBatch, const float *map,
            uint32_t mStride, size_t mBatch)
{
    const uint32_t img = blockIdx.z;
    const int x = blockIdx.x * WF_BX + threadIdx.x;
    for (int r = 0; r < WF_ROWS; r++) {
        const int y = blockIdx.y * WF_TILE_H + r * WF_BY + threadIdx.y;
        if (x >= (int)dw || y >= (int)dh) continue;
        const float *m = (const float *)((const uint8_t *)map + img * mBatch + (size_t)y * mStride) + 2 * x;
        ((float *)((uint8_t *)dst + img * dBatch + (size_t)y * dStride))[x] = bilinear(S, img, 0, 0, m[0], m[1]).val;
    }
}

// ------------------------------------------------------------------ adjoint kernels --------------
// workgroups reach the XCDs round robin; this mapping gives each XCD one contiguous run of tiles, so the
// 128-byte lines at the edges of a tile's source footprint are in the L2 that its neighbour already filled
MVX_DEV uint32_t xcd_order(uint32_t id, uint32_t n)
{
    const uint32_t q = n >> 3, r = n & 7u, xcd = id & 7u, k = id >> 3;
    return xcd * q + min(xcd, r) + k;
}

// sum over each row of 16 lanes by DPP lane shifts (one instruction a step): valid in the row's last lane
MVX_DEV float row16_sum(float v)
{
#define MVX_DPP_ADD(ctrl) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true))
    MVX_DPP_ADD(0x111);   // row_shr:1
    MVX_DPP_ADD(0x112);
    MVX_DPP_ADD(0x114);
    MVX_DPP_ADD(0x118);
#undef MVX_DPP_ADD
    return v;
}

// block sum of WF_SLOTS values: rows of 16 lanes in registers, then the block's 16 rows through LDS; slot k
// of tile t of image img goes to partials[(img * WF_SLOTS + k) * tiles + t]
MVX_DEV void block_sum_store(const float (&acc)[WF_SLOTS], float *out, uint32_t tiles)
{
    constexpr int ROWS16 = WF_BX * WF_BY / 16;
    __shared__ float part[ROWS16][WF_SLOTS];
    const int tid = threadIdx.y * WF_BX + threadIdx.x;
#pragma unroll
    for (int k = 0; k < WF_SLOTS; k++) {
        const float v = row16_sum(acc[k]);
        if ((tid & 15) == 15) part[tid >> 4][k] = v;
    }
    __syncthreads();
    if (tid < WF_SLOTS) {
        float v = part[0][tid];
#pragma unroll
        for (int r = 1; r < ROWS16; r++) v += part[r][tid];
        out[(size_t)tid * tiles] = v;
    }
}

MVX_DEV bool wave_all(bool v) { return __builtin_amdgcn_ballot_w64(v) == __builtin_amdgcn_ballot_w64(true); }

// dL/dsrc of one wave's samples, taken row by row.  Four atomics a pixel were the larger part of the
// adjoint; neighbouring pixels add to the same source pixels, so they are merged in registers first: a lane
// passes its right-hand column to the next lane when that lane's cell is the next one, and keeps its lower
// row for the next image row's upper one.  Near unit scale that leaves about one atomic per pixel; samples
// that do not line up (scaled, steeply rotated) add on their own as before.  An LDS image of the block's
// footprint was measured too: its F32 LDS adds cost as much as the global atomics.
MVX_DEV int dpp_prev(int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x138, 0xf, 0xf, false); }
MVX_DEV int dpp_next(int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x130, 0xf, 0xf, false); }
MVX_DEV float dpp_prev(float v) { return __int_as_float(dpp_prev(0, __float_as_int(v))); }

struct SrcGrad {
    static constexpr int NONE = INT_MIN / 2;
    uint8_t *base;
    uint32_t stride, w, h;
    int bx = NONE, by = NONE;       // the pending lower row: pixels (bx, by) and (bx + 1, by)
    float b0 = 0.f, b1 = 0.f;

    MVX_DEV void add(int x, int y, float v)
    {
        if ((v != 0.f) & ((uint32_t)x < w) & ((uint32_t)y < h)) atomicAdd((float *)(base + (size_t)(uint32_t)y * stride) + x, v);
    }
    // one row, every lane of the wave active; lanes with `take` unset have nothing to add
    MVX_DEV void row(bool take, const Sample &s, float g)
    {
        const int x0 = take ? s.x0 : NONE, y0 = take ? s.y0 : NONE;
        const float gx = 1.f - s.fx, gy = 1.f - s.fy;
        const float w00 = gx * gy, w01 = s.fx * gy, w10 = gx * s.fy, w11 = s.fx * s.fy;
        float c00 = take && w00 != 0.f ? g * w00 : 0.f, c01 = take && w01 != 0.f ? g * w01 : 0.f;
        float c10 = take && w10 != 0.f ? g * w10 : 0.f, c11 = take && w11 != 0.f ? g * w11 : 0.f;
        const bool below = (x0 == bx) & (y0 == by);
        if (!below) { add(bx, by, b0); add(bx + 1, by, b1); }
        c00 += below ? b0 : 0.f;
        c01 += below ? b1 : 0.f;
        const int left = (dpp_prev(NONE - 1, x0) + 1 == x0) & (dpp_prev(NONE, y0) == y0) & (x0 != NONE);
        const float l0 = dpp_prev(c01), l1 = dpp_prev(c11);
        c00 += left ? l0 : 0.f;
        c10 += left ? l1 : 0.f;
        const bool given = dpp_next(0, left) != 0;
        add(x0, y0, c00);
        add(x0 + 1, y0, given ? 0.f : c01);
        bx = x0; by = y0 + 1;
        b0 = c10; b1 = given ? 0.f : c11;
    }
    MVX_DEV void finish() { add(bx, by, b0); add(bx + 1, by, b1); }
};

// MODE 0: g given per pixel (gradient of an arbitrary loss); MODE 1: L2 against `G`, g = 2 weight r.
//
// A wave owns a strip of 64 columns and ROWS consecutive rows, one row at a time.  Bound by VALU issue
// (about 90 instructions a row) and for large batches not far from memory (8 bytes a pixel).  What keeps the
// instructions down: one reciprocal serves all four quotients of a pixel; a column's X is the same in all
// of a lane's rows, so only the sums of a, b, c and of a Y, b Y, c Y are kept and the X sums formed once;
// rows whose samples all lie inside the source, in front and with z in [2^-60, 2^60] (the usual case) take
// their four pixels with two unchecked loads off one 32-bit offset, others clamped loads, and where z or a
// position is out of the ordinary the plain divisions.  The sample positions are project()'s, operation by
// operation and with quotients rounded as its divisions are, so forward and adjoint sample the same cells.
// Eight waves a SIMD hide the loads better than more loads in flight per wave: with two and four rows at a time
// (58 to 96 and 115 to 155 registers) the batch below took 236 and 286 us in all, with one row 232.
// 64 pairs of 1024x1024 and their two smaller levels (L2, no source gradient), reductions included: 417 us
// with four divisions, checked loads, ten sums a pixel and shuffle reductions; 232 us now.  With dL/dsrc, 8
// images of 509x387: 42.7 us with four atomics a pixel, 20.5 us now.
template <int MODE, int ROWS, bool SCAT>
__global__ void __launch_bounds__(WF_BX * WF_BY, SCAT ? 7 : 8)
k_warp_f32_adjoint(F32Plane S, F32Plane G, uint32_t dw, uint32_t dh, uint32_t tilesX, const double *Hs, float weight,
                   float *gsrc, uint32_t gsStride, size_t gsBatch, float *partials)
{
    const uint32_t tiles = gridDim.x * gridDim.y;   // a 1-D grid but for the largest images
    const uint32_t id = xcd_order((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, tiles * gridDim.z);
    const uint32_t img = id / tiles, tile = id - img * tiles;
    const uint32_t ty = tile / tilesX, tx = tile - ty * tilesX;
    const int yw = (int)((ty * WF_BY + __builtin_amdgcn_readfirstlane(threadIdx.y)) * ROWS);
    const int xl = (int)(tx * WF_BX + threadIdx.x);
    const bool inx = xl < (int)dw;
    const int x = min(xl, (int)dw - 1);   // lanes past the right edge repeat the last column and are left out of the sums
    const HomF H = load_hom(Hs + 9 * img);
    const float X = (float)x;
    const float q0 = H.h6 * X, u0 = H.d0 * X, v0 = H.h3 * X;
    const uint8_t *gbase = (const uint8_t *)G.p + img * G.batch, *sbase = (const uint8_t *)S.p + img * S.batch;
    // cells floor(du), floor(dv) whose four pixels lie inside the source: [lo, hi] (none when offsets or
    // coordinates outgrow 32 bits, a float or a 24-bit product)
    const bool small = max(max(dw, dh), max(S.w, S.h)) < (1u << 24) && S.stride < (1u << 24) && (uint64_t)S.h * S.stride < (1ull << 32);
    const float lox = small ? -X : INFINITY, hix = (float)((int)S.w - 2) - X, hiy = (float)((int)S.h - 2);
    float sa = 0.f, sb = 0.f, sc = 0.f, saY = 0.f, sbY = 0.f, scY = 0.f, loss = 0.f;
    SrcGrad sg{(uint8_t *)gsrc + img * gsBatch, gsStride, S.w, S.h};
#pragma unroll 1
    for (int y = yw; y < min(yw + ROWS, (int)dh); y++) {
        const float target = ((const float *)(gbase + (size_t)y * G.stride))[x];
        const float Y = (float)y;
        const float q = q0 + H.h7 * Y, z = q + H.h8;
        const float nu = (u0 + H.h1 * Y + H.h2) - X * q, nv = (v0 + H.d4 * Y + H.h5) - Y * q;
        const float rz = recip_usual(z);
        float du = div_by(nu, z, rz), dv = div_by(nv, z, rz);
        float fu = floorf(du), fv = floorf(dv);
        Sample s;
        s.ok = true;
        s.x0 = x + (int)fu; s.y0 = y + (int)fv;
        const bool usual = (z >= 0x1p-60f) & (z <= 0x1p60f);
        const auto accumulate = [&](auto check, auto quotients) {
            constexpr bool CHECK = decltype(check)::value, QUOTIENTS = decltype(quotients)::value;
            s.fx = du - fu; s.fy = dv - fv;
            const float gx = 1.f - s.fx, gy = 1.f - s.fy;
            const float Iu = fmaf(s.fy, s.p11 - s.p10, gy * (s.p01 - s.p00)), Iv = fmaf(s.fx, s.p11 - s.p01, gx * (s.p10 - s.p00));
            float g = target;
            if (MODE == 1) {
                const float top = fmaf(s.fx, s.p01, gx * s.p00), bot = fmaf(s.fx, s.p11, gx * s.p10);
                const float val = CHECK && !s.ok ? 0.f : fmaf(s.fy, bot, gy * top);
                const float res = val - g, wr = weight * res;
                loss += wr * res;
                g = 2.f * wr;
            }
            const bool take = (!CHECK || s.ok) & (g != 0.f);
            if (take) {
                // (rz, or g rz, may overflow where the quotients do not)
                const float gz = QUOTIENTS ? g : g * rz;
                const float a = QUOTIENTS ? gz * Iu / z : gz * Iu, b = QUOTIENTS ? gz * Iv / z : gz * Iv, c = -fmaf(a, X + du, b * (Y + dv));
                sa += a; sb += b; sc += c;
                saY = fmaf(a, Y, saY); sbY = fmaf(b, Y, sbY); scY = fmaf(c, Y, scY);
            }
            if (SCAT) sg.row(take & inx, s, g);
        };
        if (wave_all(usual & (fu >= lox) & (fu <= hix) & (fv >= -Y) & (fv <= hiy - Y))) {
            const uint32_t off = __umul24((uint32_t)s.y0, S.stride) + 4u * (uint32_t)s.x0;
            const float2a t = *(const float2a *)(sbase + off), b = *(const float2a *)(sbase + S.stride + off);
            s.p00 = t.x; s.p01 = t.y; s.p10 = b.x; s.p11 = b.y;
            accumulate(std::false_type(), std::false_type());
        } else {
            const bool plain = !wave_all(usual & (fabsf(du) < 1.0e7f) & (fabsf(dv) < 1.0e7f));
            if (plain) {
                du = nu / z;
                dv = nv / z;
                s.ok = (z > 0.f) & (fabsf(du) < 1.0e7f) & (fabsf(dv) < 1.0e7f);   // also false for NaN
                if (!s.ok) du = dv = 0.f;
                fu = floorf(du); fv = floorf(dv);
                s.x0 = x + (int)fu; s.y0 = y + (int)fv;
            }
            // every load inside the source, pixels outside it then 0
            const int xe = (int)S.w - 1, ye = (int)S.h - 1;
            const int xa = min(max(s.x0, 0), xe), xb = min(max(s.x0 + 1, 0), xe), ya = min(max(s.y0, 0), ye), yb = min(max(s.y0 + 1, 0), ye);
            const float *ra = (const float *)(sbase + (size_t)(uint32_t)ya * S.stride), *rb = (const float *)(sbase + (size_t)(uint32_t)yb * S.stride);
            const float t0 = ra[xa], t1 = ra[xb], t2 = rb[xa], t3 = rb[xb];
            const bool ia = xa == s.x0, ib = xb == s.x0 + 1, ja = ya == s.y0, jb = yb == s.y0 + 1;
            s.p00 = (ia & ja) ? t0 : 0.f; s.p01 = (ib & ja) ? t1 : 0.f;
            s.p10 = (ia & jb) ? t2 : 0.f; s.p11 = (ib & jb) ? t3 : 0.f;
            if (plain) accumulate(std::true_type(), std::true_type());
            else accumulate(std::true_type(), std::false_type());
        }
    }
    if (SCAT) sg.finish();
    float acc[WF_SLOTS] = {sa * X, saY, sa, sb * X, sbY, sb, sc * X, scY, sc, loss};
    if (!inx)
#pragma unroll
        for (int k = 0; k < WF_SLOTS; k++) acc[k] = 0.f;
    block_sum_store(acc, partials + (size_t)img * WF_SLOTS * tiles + tile, tiles);
}

// dH[img][0..8] (and loss[img]) = F64 sums of the per-workgroup partials, in a fixed order; one workgroup
// per image and slot (64 images, 512 partials a slot: 18 us when one workgroup took all ten slots in turn,
// 5 us now)
__global__ void __launch_bounds__(256)
k_reduce_partials(const float *partials, uint32_t blocks, double *gradH, double *loss, int accumulate)
{
    const uint32_t img = blockIdx.x, k = blockIdx.y;
    __shared__ double red[4];
    const float *p = partials + ((size_t)img * WF_SLOTS + k) * blocks;
    double v = 0.0;
    for (uint32_t b = threadIdx.x; b < blocks; b += 256) v += (double)p[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double t = ((red[0] + red[1]) + red[2]) + red[3];
        double *o = (k < 9) ? (gradH ? gradH + 9 * img + k : nullptr) : (loss ? loss + img : nullptr);
        if (o) *o = accumulate ? *o + t : t;
    }
}

__global__ void __launch_bounds__(WF_BX * WF_BY)
k_remap_f32_adjoint(F32Plane S, F32Plane G, uint32_t dw, uint32_t dh, const float *map, uint32_t mStride, size_t mBatch,
                    float *gsrc, uint32_t gsStride, size_t gsBatch, float *gmap, uint32_t gmStride, size_t gmBatch)
{
    const uint32_t img = blockIdx.z;
    const int x = blockIdx.x * WF_BX + threadIdx.x;
    for (int r = 0; r < WF_ROWS; r++) {
        const int y = blockIdx.y * WF_TILE_H + r * WF_BY + threadIdx.y;
        if (x >= (int)dw || y >= (int)dh) continue;
        const float *m = (const float *)((const uint8_t *)map + img * mBatch + (size_t)y * mStride) + 2 * x;
        const Sample s = bilinear(S, img, 0, 0, m[0], m[1]);
        const float g = row_of(G, img, y)[x];
        float gu = 0.f, gv = 0.f;
        if (s.ok) {
            gu = g * ((1.f - s.fy) * (s.p01 - s.p00) + s.fy * (s.p11 - s.p10));
            gv = g * ((1.f - s.fx) * (s.p10 - s.p00) + s.fx * (s.p11 - s.p01));
            if (gsrc && g != 0.f) scatter((float *)((uint8_t *)gsrc + img * gsBatch), gsStride, S.w, S.h, s, g);
        }
        if (gmap) {
            float *o = (float *)((uint8_t *)gmap + img * gmBatch + (size_t)y * gmStride) + 2 * x;
            o[0] = gu;
            o[1] = gv;
        }
    }
}

// ------------------------------------------------------------------ F32 pyramid --------------------
// out(x, y) = sum_{i,j} w_i w_j in(clamp(2x+i-2), clamp(2y+j-2)) / 256, w = [1 4 6 4 1]
__constant__ float kPyrW[5] = {1.f, 4.f, 6.f, 4.f, 1.f};

__global__ void __launch_bounds__(WF_BX * WF_BY)
k_pyr_half_f32(F32Plane S, float *dst, uint32_t dw, uint32_t dh, uint32_t dStride, size_t dBatch)
{
    const uint32_t img = blockIdx.z;
    const int x = blockIdx.x * WF_BX + threadIdx.x;
    for (int r = 0; r < WF_ROWS; r++) {
        const int y = blockIdx.y * WF_TILE_H + r * WF_BY + threadIdx.y;
        if (x >= (int)dw || y >= (int)dh) continue;
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < 5; j++) {
            const int sy = min(max(2 * y + j - 2, 0), (int)S.h - 1);
            const float *row = row_of(S, img, sy);
            float hs = 0.f;
#pragma unroll
            for (int i = 0; i < 5; i++) hs += kPyrW[i] * row[min(max(2 * x + i - 2, 0), (int)S.w - 1)];
            acc += kPyrW[j] * hs;
        }
        ((float *)((uint8_t *)dst + img * dBatch + (size_t)y * dStride))[x] = acc * (1.f / 256.f);
    }
}

// weight with which output column x (of n_out) reads input column X (of n_in): taps whose clamped
// position is X
MVX_DEV float tap_weight(int x, int X, int n_in)
{
    float w = 0.f;
#pragma unroll
    for (int i = 0; i < 5; i++) w += (min(max(2 * x + i - 2, 0), n_in - 1) == X) ? kPyrW[i] : 0.f;
    return w;
}

// gradSrc(X, Y) += sum over the outputs that read it (a gather: no atomics)
__global__ void __launch_bounds__(WF_BX * WF_BY)
k_pyr_half_f32_adjoint(F32Plane G, float *gsrc, uint32_t sw, uint32_t sh, uint32_t gsStride, size_t gsBatch)
{
    const uint32_t img = blockIdx.z;
    const int X = blockIdx.x * WF_BX + threadIdx.x;
    for (int r = 0; r < WF_ROWS; r++) {
        const int Y = blockIdx.y * WF_TILE_H + r * WF_BY + threadIdx.y;
        if (X >= (int)sw || Y >= (int)sh) continue;
        float acc = 0.f;
        for (int y = (Y >> 1) - 1; y <= (Y >> 1) + 1; y++) {
            if (y < 0 || y >= (int)G.h) continue;
            const float wy = tap_weight(y, Y, (int)sh);
            if (wy == 0.f) continue;
            const float *row = row_of(G, img, y);
            float hs = 0.f;
            for (int x = (X >> 1) - 1; x <= (X >> 1) + 1; x++) {
                if (x < 0 || x >= (int)G.w) continue;
                hs += tap_weight(x, X, (int)sw) * row[x];
            }
            acc += wy * hs;
        }
        float *o = (float *)((uint8_t *)gsrc + img * gsBatch + (size_t)Y * gsStride) + X;
        *o += acc * (1.f / 256.f);
    }
}

inline bool f32_plane_ok(const void *p, uint32_t w, uint32_t h, uint32_t stride, size_t batch, uint32_t count, uint32_t floats = 1)
{
    if (!p || (reinterpret_cast<uintptr_t>(p) & 3u) || w == 0 || h == 0) return false;
    if (stride < w * 4u * floats || (stride & 3u)) return false;
    if (count > 1 && (batch < (size_t)stride * h || (batch & 3u))) return false;
    return true;
}

inline dim3 f32_grid(uint32_t w, uint32_t h, uint32_t count)
{
    return dim3((w + WF_TILE_W - 1) / WF_TILE_W, (h + WF_TILE_H - 1) / WF_TILE_H, count);
}

}  // namespace mvx

using namespace mvx;

extern "C" int mvx_WarpPerspective_F32_Bilinear(mvx_stream_t stream, uint32_t count, uint32_t dw, uint32_t dh, float *dst,
                                                uint32_t dstStride, size_t dstBatchStride, uint32_t sw, uint32_t sh,
                                                const float *src, uint32_t srcStride, size_t srcBatchStride, const double *H)
{
    if (count == 0) return MVX_SUCCESS;
    if (!f32_plane_ok(dst, dw, dh, dstStride, dstBatchStride, count) || !f32_plane_ok(src, sw, sh, srcStride, srcBatchStride, count) ||
        !H || count > 65535)
        return MVX_ERROR_INVALID_PARAMETERS;
    const F32Plane S{src, sw, sh, srcStride, srcBatchStride};
    hipLaunchKernelGGL(k_warp_f32, f32_grid(dw, dh, count), dim3(WF_BX, WF_BY), 0, stream_of(stream), S, dst, dw, dh, dstStride,
                       dstBatchStride, H);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" size_t mvx_warp_perspective_f32_workspace_size(uint32_t count, uint32_t dw, uint32_t dh)
{
    const dim3 g = f32_grid(dw, dh, count);
    return (size_t)g.x * g.y * count * WF_SLOTS * sizeof(float);
}

static int warp_adjoint_common(mvx_stream_t stream, int mode, uint32_t count, uint32_t dw, uint32_t dh, const float *g,
                               uint32_t gStride, size_t gBatch, uint32_t sw, uint32_t sh, const float *src, uint32_t srcStride,
                               size_t srcBatch, const double *H, float weight, double *loss, double *gradH, float *gradSrc,
                               uint32_t gsStride, size_t gsBatch, int accumulate, void *ws, size_t wsSize)
{
    if (count == 0) return MVX_SUCCESS;
    if (!f32_plane_ok(g, dw, dh, gStride, gBatch, count) || !f32_plane_ok(src, sw, sh, srcStride, srcBatch, count) || !H ||
        count > 65535)
        return MVX_ERROR_INVALID_PARAMETERS;
    if (gradSrc && !f32_plane_ok(gradSrc, sw, sh, gsStride, gsBatch, count)) return MVX_ERROR_INVALID_PARAMETERS;
    if (!ws || (reinterpret_cast<uintptr_t>(ws) & 3u) || wsSize < mvx_warp_perspective_f32_workspace_size(count, dw, dh))
        return MVX_ERROR_INVALID_PARAMETERS;
    const F32Plane S{src, sw, sh, srcStride, srcBatch}, G{g, dw, dh, gStride, gBatch};
    float *part = (float *)ws;
    const uint32_t tilesX = (dw + WF_BX - 1) / WF_BX;
    const auto tiles_of = [&](uint32_t rows) { return (uint64_t)tilesX * ((dh + WF_BY * rows - 1) / (WF_BY * rows)); };
    // rows per wave: setup and block sum cost about 100 instructions a wave, so eight rows where that leaves
    // two rounds of waves or more for the 1024 SIMDs, else four (sixteen was no faster for 64 x 1024x1024)
    const uint32_t rows = tiles_of(8) * count >= 2048 ? 8 : 4;
    const uint64_t tiles = tiles_of(rows);
    if (tiles * count > 0xffffffffull) return MVX_ERROR_INVALID_PARAMETERS;   // the kernel's 32-bit tile numbers
    // a launch takes below 2^32 threads in x; images of more than 34 Gpixel have a row of tiles there
    const dim3 grid = tiles <= 0xffffffull ? dim3((uint32_t)tiles, 1, count) : dim3(tilesX, (uint32_t)(tiles / tilesX), count);
    const auto run = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(WF_BX, WF_BY), 0, stream_of(stream), S, G, dw, dh, tilesX, H, weight,
                           gradSrc, gsStride, gsBatch, part);
    };
    const auto pick = [&](auto m) {
        constexpr int M = decltype(m)::value;
        if (gradSrc) rows == 8 ? run(k_warp_f32_adjoint<M, 8, true>) : run(k_warp_f32_adjoint<M, 4, true>);
        else rows == 8 ? run(k_warp_f32_adjoint<M, 8, false>) : run(k_warp_f32_adjoint<M, 4, false>);
    };
    if (mode == 1) pick(std::integral_constant<int, 1>());
    else pick(std::integral_constant<int, 0>());
    MVX_LAUNCH_CHECK();
    if (gradH || loss) {
        hipLaunchKernelGGL(k_reduce_partials, dim3(count, WF_SLOTS), dim3(256), 0, stream_of(stream), part, (uint32_t)tiles, gradH,
                           loss, accumulate);
        MVX_LAUNCH_CHECK();
    }
    return MVX_SUCCESS;
}

extern "C" int mvx_warp_perspective_f32_adjoint(mvx_stream_t stream, uint32_t count, uint32_t dw, uint32_t dh, const float *gradOut,
                                                uint32_t gStride, size_t gBatchStride, uint32_t sw, uint32_t sh, const float *src,
                                                uint32_t srcStride, size_t srcBatchStride, const double *H, float *gradSrc,
                                                uint32_t gsStride, size_t gsBatchStride, double *gradH, void *workspace,
                                                size_t workspaceSize)
{
    return warp_adjoint_common(stream, 0, count, dw, dh, gradOut, gStride, gBatchStride, sw, sh, src, srcStride, srcBatchStride, H,
                               1.f, nullptr, gradH, gradSrc, gsStride, gsBatchStride, 0, workspace, workspaceSize);
}

extern "C" int mvx_warp_perspective_f32_l2(mvx_stream_t stream, uint32_t count, uint32_t dw, uint32_t dh, const float *target,
                                           uint32_t tStride, size_t tBatchStride, uint32_t sw, uint32_t sh, const float *src,
                                           uint32_t srcStride, size_t srcBatchStride, const double *H, float weight, double *loss,
                                           double *gradH, float *gradSrc, uint32_t gsStride, size_t gsBatchStride, int accumulate,
                                           void *workspace, size_t workspaceSize)
{
    return warp_adjoint_common(stream, 1, count, dw, dh, target, tStride, tBatchStride, sw, sh, src, srcStride, srcBatchStride, H,
                               weight, loss, gradH, gradSrc, gsStride, gsBatchStride, accumulate, workspace, workspaceSize);
}

extern "C" int mvx_Remap_F32_Bilinear(mvx_stream_t stream, uint32_t count, uint32_t dw, uint32_t dh, float *dst, uint32_t dstStride,
                                      size_t dstBatchStride, uint32_t sw, uint32_t sh, const float *src, uint32_t srcStride,
                                      size_t srcBatchStride, const float *map, uint32_t mapStride, size_t mapBatchStride)
{
    if (count == 0) return MVX_SUCCESS;
    if (!f32_plane_ok(dst, dw, dh, dstStride, dstBatchStride, count) || !f32_plane_ok(src, sw, sh, srcStride, srcBatchStride, count) ||
        !f32_plane_ok(map, dw, dh, mapStride, mapBatchStride, count, 2) || count > 65535)
        return MVX_ERROR_INVALID_PARAMETERS;
    const F32Plane S{src, sw, sh, srcStride, srcBatchStride};
    hipLaunchKernelGGL(k_remap_f32, f32_grid(dw, dh, count), dim3(WF_BX, WF_BY), 0, stream_of(stream), S, dst, dw, dh, dstStride,
                       dstBatchStride, map, mapStride, mapBatchStride);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" int mvx_remap_f32_adjoint(mvx_stream_t stream, uint32_t count, uint32_t dw, uint32_t dh, const float *gradOut,
                                     uint32_t gStride, size_t gBatchStride, uint32_t sw, uint32_t sh, const float *src,
                                     uint32_t srcStride, size_t srcBatchStride, const float *map, uint32_t mapStride,
                                     size_t mapBatchStride, float *gradSrc, uint32_t gsStride, size_t gsBatchStride, float *gradMap,
                                     uint32_t gmStride, size_t gmBatchStride)
{
    if (count == 0) return MVX_SUCCESS;
    if (!f32_plane_ok(gradOut, dw, dh, gStride, gBatchStride, count) || !f32_plane_ok(src, sw, sh, srcStride, srcBatchStride, count) ||
        !f32_plane_ok(map, dw, dh, mapStride, mapBatchStride, count, 2) || count > 65535)
        return MVX_ERROR_INVALID_PARAMETERS;
    if (gradSrc && !f32_plane_ok(gradSrc, sw, sh, gsStride, gsBatchStride, count)) return MVX_ERROR_INVALID_PARAMETERS;
    if (gradMap && !f32_plane_ok(gradMap, dw, dh, gmStride, gmBatchStride, count, 2)) return MVX_ERROR_INVALID_PARAMETERS;
    const F32Plane S{src, sw, sh, srcStride, srcBatchStride}, G{gradOut, dw, dh, gStride, gBatchStride};
    hipLaunchKernelGGL(k_remap_f32_adjoint, f32_grid(dw, dh, count), dim3(WF_BX, WF_BY), 0, stream_of(stream), S, G, dw, dh, map,
                       mapStride, mapBatchStride, gradSrc, gsStride, gsBatchStride, gradMap, gmStride, gmBatchStride);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" int mvx_PyramidHalf_F32(mvx_stream_t stream, uint32_t count, uint32_t dw, uint32_t dh, float *dst, uint32_t dstStride,
                                   size_t dstBatchStride, uint32_t sw, uint32_t sh, const float *src, uint32_t srcStride,
                                   size_t srcBatchStride)
{
    if (count == 0) return MVX_SUCCESS;
    if (dw != (sw + 1) / 2 || dh != (sh + 1) / 2 || !f32_plane_ok(dst, dw, dh, dstStride, dstBatchStride, count) ||
        !f32_plane_ok(src, sw, sh, srcStride, srcBatchStride, count) || count > 65535)
        return MVX_ERROR_INVALID_PARAMETERS;
    const F32Plane S{src, sw, sh, srcStride, srcBatchStride};
    hipLaunchKernelGGL(k_pyr_half_f32, f32_grid(dw, dh, count), dim3(WF_BX, WF_BY), 0, stream_of(stream), S, dst, dw, dh, dstStride,
                       dstBatchStride);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" int mvx_pyramid_half_f32_adjoint(mvx_stream_t stream, uint32_t count, uint32_t sw, uint32_t sh, float *gradSrc,
                                            uint32_t gsStride, size_t gsBatchStride, uint32_t dw, uint32_t dh, const float *gradDst,
                                            uint32_t gStride, size_t gBatchStride)
{
    if (count == 0) return MVX_SUCCESS;
    if (dw != (sw + 1) / 2 || dh != (sh + 1) / 2 || !f32_plane_ok(gradSrc, sw, sh, gsStride, gsBatchStride, count) ||
        !f32_plane_ok(gradDst, dw, dh, gStride, gBatchStride, count) || count > 65535)
        return MVX_ERROR_INVALID_PARAMETERS;
    const F32Plane G{gradDst, dw, dh, gStride, gBatchStride};
    hipLaunchKernelGGL(k_pyr_half_f32_adjoint, f32_grid(sw, sh, count), dim3(WF_BX, WF_BY), 0, stream_of(stream), G, gradSrc, sw, sh,
                       gsStride, gsBatchStride);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}
