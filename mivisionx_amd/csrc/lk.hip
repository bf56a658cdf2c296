// lk.hip -- pyramidal Lucas-Kanade feature tracking (OpticalFlowPyrLK_XY_XY) for gfx950.
//
// HafCpu_OpticalFlowPyrLK_XY_XY_Generic (ago_haf_cpu_opticalflow.cpp:153-546) runs on the CPU only
// in the reference (ago_kernel_api.cpp:20642-20646).  Here:
//   k_lk_scharr  per level, coarse to fine: the Scharr derivative image of the old level
//                (ComputeSharr, :59-150) and the state the reference's row scratch keeps after it;
//   k_lk_track   one 64-lane workgroup per keypoint takes the point through the levels: patch
//                extraction, the 2x2 structure tensor, and the Newton iterations against the new level.
// Results are bit-identical to the reference:
//   * the reference keeps a row scratch B (u16: trow0 = B, trow1 = B + ceil8(W+2)) and the
//     derivative image D (stride = level-0 width) in the node's zero-initialised local data, and
//     reads cells of them that only earlier levels or earlier calls wrote (B[-1], B[W8],
//     B[ceil8(W+2)-1], B[ceil8(W+2)+W8]; D columns >= W8 and row 0, W8 = W & ~7).  The workspace
//     here holds the same B, D and per-point positions with the same life time, so successive
//     calls reproduce the reference's successive calls;
//   * float sums follow the reference's SSE order: per-lane partial sums over 4- or 8-column
//     groups, rows in order, scalar columns separately, combined as the reference writes it; the
//     b-vector scalar part accumulates in double;
//   * x86 conversions (truncation, 0x80000000 out of int32 range) are reproduced explicitly.
// The ordered sums are done by a handful of lanes reading per-pixel products from LDS; every other
// step is spread over the 64 lanes of the workgroup.
#include "mvx_common.hpp"
#include "pick.hpp"   // Keypoint (vx_keypoint_t)

namespace mvx {

namespace {

constexpr int LK_THREADS = 64;
constexpr int LK_MAX_WIN = 15;
constexpr int LK_SMALL_WIN = 11;   // windows up to here take two window pixels per lane, larger ones four
constexpr int W_BITS = 14;
constexpr uint32_t TERM_EPSILON = 0xF001, TERM_BOTH = 0xF002;   // VX_TERM_CRITERIA_*
constexpr uint32_t LK_EPS_ITER_CAP = 10000;                      // EPSILON-only has no bound in the reference

MVX_DEV int32_t x86_int(float v)
{
    if (!(v > -2147483904.0f && v < 2147483648.0f)) return INT32_MIN;
    return (int32_t)v;
}

MVX_DEV int32_t sat16(int32_t v) { return min(max(v, -32768), 32767); }

MVX_DEV int32_t descale(int32_t x, int n) { return (x + (1 << (n - 1))) >> n; }

}  // namespace

struct LkLevel {
    const uint8_t *oldImg, *newImg;
    uint32_t width, height, oldStride, newStride;
};

// 8 and 16 bytes at any address the plane's rows put them at
struct __attribute__((packed, aligned(1))) Bytes8 { uint32_t lo, hi; };
struct __attribute__((packed, aligned(4))) Words4 { uint32_t x, y, z, w; };

// ComputeSharr for rows 1..H-2, columns 0..W8-1 of the old level; neighbours outside [0, W8) come
// from the row scratch B exactly as the reference's loops read them.  The last row's threads leave in B what
// the reference's scratch holds after a level, the vertical sums of row H-2: cells [0, W8) and [T1, T1+W8),
// none of which this level reads (B[-1], B[W8], B[T1-1], B[T1+W8] with T1 >= W+2).
// `stale` (the derivative image the previous call left, or null): this level has a D of its own, and the
// cells no level writes -- row 0 and the columns from W8 on -- are copied from there; the reference has one D
// for all levels, where those cells still hold the previous call's.
// Eight columns a thread, three 8-byte loads and two 16-byte stores: bound by the 5 bytes a pixel it moves
// (3840x2160: one column a thread, byte loads 32 us; 14 us now).
__global__ void __launch_bounds__(256)
k_lk_scharr(LkLevel L, int16_t *__restrict__ D, uint32_t dStride, uint16_t *B, const int16_t *stale, uint32_t staleStride)
{
    const uint32_t W8 = L.width & ~7u, T1 = (L.width + 2u + 7u) & ~7u;
    const uint32_t x0 = (blockIdx.x * 64 + threadIdx.x) * 8;
    const uint32_t y = 1 + blockIdx.y * 4 + threadIdx.y;
    if (x0 > W8 || y + 1 >= L.height) return;
    if (x0 == W8) {
        if (stale)
            for (uint32_t x = W8; x < L.width; x++)
                for (int k = 0; k < 2; k++) D[(uint64_t)y * dStride + 2 * x + k] = stale[(uint64_t)y * staleStride + 2 * x + k];
        return;
    }
    if (stale && y == 1)
        for (uint32_t i = 2 * x0; i < (x0 + 8 == W8 ? 2 * L.width : 2 * x0 + 16); i++) D[i] = stale[i];
    const uint8_t *r0 = L.oldImg + (uint64_t)(y - 1) * L.oldStride + x0, *r1 = r0 + L.oldStride, *r2 = r1 + L.oldStride;
    const Bytes8 v0 = *(const Bytes8 *)r0, v1 = *(const Bytes8 *)r1, v2 = *(const Bytes8 *)r2;
    int32_t t0[10], t1[10];   // columns x0-1 .. x0+8
    auto sums = [&](int i, int32_t p0, int32_t p1, int32_t p2) { t0[i] = (p0 + p2) * 3 + p1 * 10; t1[i] = p2 - p0; };
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int sh = 8 * (i & 3);
        sums(i + 1, (int32_t)(((i < 4 ? v0.lo : v0.hi) >> sh) & 0xffu), (int32_t)(((i < 4 ? v1.lo : v1.hi) >> sh) & 0xffu),
             (int32_t)(((i < 4 ? v2.lo : v2.hi) >> sh) & 0xffu));
    }
    if (x0 == 0) { t0[0] = (int32_t)B[-1]; t1[0] = (int32_t)(int16_t)B[T1 - 1]; }
    else sums(0, r0[-1], r1[-1], r2[-1]);
    if (x0 + 8 == W8) { t0[9] = (int32_t)B[W8]; t1[9] = (int32_t)(int16_t)B[T1 + W8]; }
    else sums(9, r0[8], r1[8], r2[8]);
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t gx = (uint32_t)(t0[i + 2] - t0[i]), gy = (uint32_t)((t1[i] + t1[i + 2]) * 3 + t1[i + 1] * 10);
        o[i] = (gx & 0xffffu) | (gy << 16);
    }
    Words4 *d = (Words4 *)(D + (uint64_t)y * dStride + 2ull * x0);
    d[0] = Words4{o[0], o[1], o[2], o[3]};
    d[1] = Words4{o[4], o[5], o[6], o[7]};
    if (y + 2 == L.height)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            B[x0 + i] = (uint16_t)t0[i + 1];
            B[T1 + x0 + i] = (uint16_t)t1[i + 1];
        }
}

// sum of an F64 over the wave by DPP lane shifts, in every lane (no LDS round trips: six shuffles of a double
// took longer than an iteration's arithmetic)
template <int CTRL, int ROWS> MVX_DEV double dpp_add(double v)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

MVX_DEV double wave_sum(double v)
{
    v = dpp_add<0x111, 0xf>(v);
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);   // lane 15 of each row of 16 holds the row's sum
    v = dpp_add<0x142, 0xa>(v);   // rows 0 and 2 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);   // rows 0 and 1 into rows 2 and 3: lane 63 holds them all
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 63), hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 63);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

constexpr uint32_t LK_MAX_LEVELS = 16;

struct LkTrackLevel {
    LkLevel img;
    const int16_t *D;
    uint32_t dStride;
    float ptScale;
};

struct LkParams {
    uint32_t first, last, levels;   // levels first, first-1, .. last of `levels`
    uint32_t winsz, halfWin, iterations, termination, useEstimate;
    float epsilon;
    LkTrackLevel level[LK_MAX_LEVELS];
};

// a point's state between levels
struct LkPoint {
    Keypoint *nk;
    float x, y;          // position before the level's window offset (the reference's next point)
    int32_t status;
};

// one level of one point, the whole wave; sI.. are npix long, sAcc 24
template <int MAXW>
MVX_DEV void lk_level(const LkParams &P, uint32_t lev, const Keypoint &ok, LkPoint &pt, int32_t *sI, int32_t *sIx, int32_t *sIy, float *sP0,
                      float *sP1, float *sP2, float *sAcc)
{
    constexpr int PPL = (MAXW * MAXW + 63) / 64;   // window pixels per lane
    const LkLevel &L = P.level[lev].img;
    const int16_t *D = P.level[lev].D;
    const uint32_t tid = threadIdx.x;
    Keypoint *nk = pt.nk;
    const float ptScale = P.level[lev].ptScale;
    const bool finest = lev == 0;
    float nextx = pt.x, nexty = pt.y;
    float prevx = (float)ok.x * ptScale, prevy = (float)ok.y * ptScale;
    const int winsz = (int)P.winsz, npix = winsz * winsz;
    const float hw = (float)P.halfWin;
    prevx = prevx - hw;
    prevy = prevy - hw;
    nextx = nextx - hw;
    nexty = nexty - hw;
    const int32_t ipx = x86_int(floorf(prevx)), ipy = x86_int(floorf(prevy));
    const uint32_t dWidth = L.width - 2u, dHeight = L.height - 2u;
    if ((ipx < 0) | (ipx >= (int32_t)(dWidth - P.winsz)) | (ipy < 0) | (ipy >= (int32_t)(dHeight - P.winsz))) {
        if (finest && tid == 0) { nk->x = x86_int(nextx); nk->y = x86_int(nexty); nk->tracking_status = 0; nk->error = 0; }
        return;
    }
    float a = prevx - (float)ipx, b = prevy - (float)ipy;
    const uint32_t IStride = L.oldStride, JStride = L.newStride, dS = P.level[lev].dStride;
    const bool plain = (a == 0.0f) && (b == 0.0f);
    // ---- patch of the old image and its derivatives, and their products
    {
        const int iw00 = (int)((double)(((1.f - a) * (1.f - b)) * (float)(1 << W_BITS)) + 0.5);
        const int iw01 = (int)((double)((a * (1.f - b)) * (float)(1 << W_BITS)) + 0.5);
        const int iw10 = (int)((double)(((1.f - a) * b) * (float)(1 << W_BITS)) + 0.5);
        const int iw11 = (1 << W_BITS) - iw00 - iw01 - iw10;
        const int nA = winsz >= 4 ? (winsz - 4) / 4 + 1 : 0;   // SSE column groups of the interpolated path
        for (int p = (int)tid; p < npix; p += LK_THREADS) {
            const int y = p / winsz, x = p % winsz;
            const uint8_t *src = L.oldImg + (uint64_t)(y + ipy) * IStride + (ipx + x);
            const int16_t *ds = D + (uint64_t)(y + ipy) * dS + 2ull * (ipx + x);
            int32_t iv, ix, iy;
            if (plain) {
                iv = (int32_t)src[0] << 5;
                ix = ds[0];
                iy = ds[1];
            } else {
                iv = descale(src[0] * iw00 + src[1] * iw01 + src[IStride] * iw10 + src[IStride + 1] * iw11, W_BITS - 5);
                ix = descale(ds[0] * iw00 + ds[2] * iw01 + ds[dS] * iw10 + ds[dS + 2] * iw11, W_BITS);
                iy = descale(ds[1] * iw00 + ds[3] * iw01 + ds[dS + 1] * iw10 + ds[dS + 3] * iw11, W_BITS);
                if (x < 4 * nA) {   // the SSE columns saturate to int16 (packs_epi32)
                    iv = sat16(iv);
                    ix = sat16(ix);
                    iy = sat16(iy);
                }
            }
            sI[p] = (int32_t)(int16_t)iv;
            sIx[p] = (int32_t)(int16_t)ix;
            sIy[p] = (int32_t)(int16_t)iy;
            sP0[p] = (float)(ix * ix);
            sP1[p] = (float)(ix * iy);
            sP2[p] = (float)(iy * iy);
        }
        __syncthreads();
        if (plain) {
            // A += (float)(sum of 4 integer products) per group of x < winsz-4 step 4, then scalar columns
            if (tid < 3) {
                const int32_t *U = (tid == 1) ? sIx : (tid == 2 ? sIy : sIx);
                const int32_t *V = (tid == 0) ? sIx : sIy;
                float acc = 0.0f;
                for (int y = 0; y < winsz; y++) {
                    int x = 0;
                    for (; x < winsz - 4; x += 4) {
                        int32_t s = 0;
                        for (int k = 0; k < 4; k++) s += U[y * winsz + x + k] * V[y * winsz + x + k];
                        acc += (float)s;
                    }
                    for (; x < winsz; x++) acc += (float)(U[y * winsz + x] * V[y * winsz + x]);
                }
                sAcc[tid] = acc * (1.0f / (1 << 20));
            }
        } else {
            // 12 lanes: the 4 SSE lanes of A11, A12, A22; 3 lanes: the scalar columns
            if (tid < 12) {
                const int q = (int)tid / 4, k = (int)tid % 4;
                const float *Pq = q == 0 ? sP0 : (q == 1 ? sP1 : sP2);
                float acc = 0.0f;
                for (int y = 0; y < winsz; y++)
                    for (int g = 0; g < nA; g++) acc = acc + Pq[y * winsz + 4 * g + k];
                sAcc[4 + tid] = acc;
            } else if (tid < 15) {
                const int q = (int)tid - 12;
                const float *Pq = q == 0 ? sP0 : (q == 1 ? sP1 : sP2);
                float acc = 0.0f;
                for (int y = 0; y < winsz; y++)
                    for (int x = 4 * nA; x < winsz; x++) acc += Pq[y * winsz + x];
                sAcc[16 + q] = acc;
            }
            __syncthreads();
            if (tid < 3) {
                float acc = sAcc[16 + tid];
                if (winsz >= 4) acc += ((sAcc[4 + 4 * tid] + sAcc[5 + 4 * tid]) + sAcc[6 + 4 * tid]) + sAcc[7 + 4 * tid];
                sAcc[tid] = acc * (1.0f / (1 << 20));
            }
        }
        __syncthreads();
    }
    const float A11 = sAcc[0], A12 = sAcc[1], A22 = sAcc[2];
    float Dt = A11 * A22 - A12 * A12;
    const float minEig = (A22 + A11 - sqrtf((A11 - A22) * (A11 - A22) + 4.f * A12 * A12)) / (float)(2 * winsz * winsz);
    if (minEig < 1.0e-04F || Dt < 1.0e-07F) {
        if (finest && tid == 0) { nk->x = x86_int(nextx); nk->y = x86_int(nexty); nk->tracking_status = 0; nk->error = 0; }
        return;
    }
    Dt = 1.f / Dt;
    // this lane's window pixels tid + 64q: row and column (-1: none)
    int pixY[PPL], pixX[PPL];
#pragma unroll
    for (int q = 0; q < PPL; q++) {
        const int p = (int)tid + q * LK_THREADS;
        pixY[q] = p < npix ? p / winsz : -1;
        pixX[q] = p < npix ? p % winsz : 0;
    }
    float prevDx = 0.f, prevDy = 0.f, ddx = 0.f, ddy = 0.f;
    const int nB = winsz >= 8 ? (winsz - 8) / 8 + 1 : 0;   // SSE column groups of 8 in the iterations
    for (uint32_t j = 0; (j < P.iterations || P.termination == TERM_EPSILON) && j < LK_EPS_ITER_CAP;) {
        const int32_t inx = x86_int(floorf(nextx)), iny = x86_int(floorf(nexty));
        if ((inx < 0) | (inx >= (int32_t)(L.width - P.winsz)) | (iny < 0) | (iny >= (int32_t)(L.height - P.winsz))) {
            if (finest && tid == 0) { nk->tracking_status = 0; nk->error = 0; }
            break;
        }
        a = nextx - (float)inx;
        b = nexty - (float)iny;
        const int iw00 = (int)((double)(((1.f - a) * (1.f - b)) * (float)(1 << W_BITS)) + 0.5);
        const int iw01 = (int)((double)((a * (1.f - b)) * (float)(1 << W_BITS)) + 0.5);
        const int iw10 = (int)((double)(((1.f - a) * b) * (float)(1 << W_BITS)) + 0.5);
        const int iw11 = (1 << W_BITS) - iw00 - iw01 - iw10;
        // The scalar columns' terms go straight into per-lane double sums.  Each term is a float holding an
        // integer below 2^31 in magnitude (|Ix| <= 32767 times |diff| <= 40928), and there are at most
        // 15 * 7 of them, so every partial sum is an integer below 2^38: the double sums are exact in any
        // order and equal the reference's row-major loop.
        // the lane's pixels' four source bytes are all loaded before any is used
        double sx = 0.0, sy = 0.0;
        uint32_t j00[PPL], j01[PPL], j10[PPL], j11[PPL];
#pragma unroll
        for (int q = 0; q < PPL; q++) {
            j00[q] = j01[q] = j10[q] = j11[q] = 0u;
            if (pixY[q] >= 0) {
                const uint8_t *J = L.newImg + (uint64_t)(pixY[q] + iny) * JStride + (inx + pixX[q]);
                j00[q] = J[0];
                j01[q] = J[1];
                j10[q] = J[JStride];
                j11[q] = J[JStride + 1];
            }
        }
#pragma unroll
        for (int q = 0; q < PPL; q++) {
            if (pixY[q] < 0) continue;
            const int p = (int)tid + q * LK_THREADS, x = pixX[q];
            int32_t t = descale((int32_t)j00[q] * iw00 + (int32_t)j01[q] * iw01 + (int32_t)j10[q] * iw10 + (int32_t)j11[q] * iw11,
                                W_BITS - 5);
            int32_t diff;
            if (x < 8 * nB) diff = sat16(sat16(t) - sI[p]);   // packs_epi32 then subs_epi16
            else diff = t - sI[p];
            const float f0 = (float)(sIx[p] * diff), f1 = (float)(sIy[p] * diff);
            if (x < 8 * nB) {
                sP0[p] = f0;
                sP1[p] = f1;
            } else {
                sx += (double)f0;
                sy += (double)f1;
            }
        }
        static_assert(LK_THREADS == 64, "the scalar-column sums are one wave's");
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        __syncthreads();
        if (tid < 8) {
            // qb0 lanes k: x-pair (k/2) and (4 + k/2); qb1 lanes: +2; even k: Ix, odd k: Iy.  Windows of at
            // most 15 columns have at most one group of 8 (nB <= 1); the lane's terms are read first and
            // then added in the reference's order.
            static_assert(MAXW < 16, "one SSE group of 8 columns per row");
            const int arr = (int)tid / 4, k = (int)tid % 4;
            const float *Pq = (k & 1) ? sP1 : sP0;
            const int c0 = 2 * arr + k / 2;
            float acc = 0.0f;
            if (nB) {
                float v0[MAXW], v1[MAXW];
#pragma unroll
                for (int y = 0; y < MAXW; y++) {
                    v0[y] = y < winsz ? Pq[y * winsz + c0] : 0.0f;
                    v1[y] = y < winsz ? Pq[y * winsz + 4 + c0] : 0.0f;
                }
#pragma unroll
                for (int y = 0; y < MAXW; y++) {
                    if (y < winsz) {
                        acc = acc + v0[y];
                        acc = acc + v1[y];
                    }
                }
            }
            sAcc[4 + tid] = acc;
        }
        __syncthreads();
        double ib1 = sx, ib2 = sy;
        if (winsz >= 8) {
            const float bb0 = sAcc[4] + sAcc[8], bb1 = sAcc[5] + sAcc[9], bb2 = sAcc[6] + sAcc[10], bb3 = sAcc[7] + sAcc[11];
            ib1 += (double)(bb0 + bb2);
            ib2 += (double)(bb1 + bb3);
        }
        const float b1 = (float)(ib1 * (double)(1.0f / (1 << 20))), b2 = (float)(ib2 * (double)(1.0f / (1 << 20)));
        const float dx = (A12 * b2 - A22 * b1) * Dt;
        const float dy = (A12 * b1 - A11 * b2) * Dt;
        nextx += dx;
        nexty += dy;
        __syncthreads();   // sP0/sP1/sAcc are rewritten by the next iteration
        if ((dx * dx + dy * dy) <= P.epsilon && (P.termination == TERM_EPSILON || P.termination == TERM_BOTH)) break;
        if (j > 0 && (double)fabsf(dx + prevDx) < 0.01 && (double)fabsf(dy + prevDy) < 0.01) {
            ddx = dx * 0.5f;
            ddy = dy * 0.5f;
            break;
        }
        prevDx = dx;
        prevDy = dy;
        j++;
    }
    if (finest) {
        if (tid == 0) {
            nk->x = x86_int(nextx + hw - ddx + 0.5f);
            nk->y = x86_int(nexty + hw - ddy + 0.5f);
        }
    } else {
        pt.x = nextx + hw - ddx;
        pt.y = nexty + hw - ddy;
    }
}

// One point through levels P.first .. P.last.  All levels in one launch where the workspace holds a
// derivative image per level: a launch lasts as long as its slowest point, and few points are slow at
// every level (10,000 points in 3840x2160, four levels: 4 x 51 us a level at a time, 110 us in one launch).
// Otherwise one launch per level, the positions kept in `next` between them.
template <int MAXW>
__global__ void __launch_bounds__(LK_THREADS)
k_lk_track(LkParams P, float2 *__restrict__ next, const Keypoint *__restrict__ oldKp, const Keypoint *__restrict__ estKp,
           Keypoint *__restrict__ newKp, const uint32_t *__restrict__ oldCount, uint32_t *__restrict__ newCount, uint32_t capacity)
{
    extern __shared__ int32_t lds[];   // 6 npix + 24 words
    const uint32_t tid = threadIdx.x;
    const uint32_t id = blockIdx.x;
    const uint32_t n = min(*oldCount, capacity);
    if (P.last == 0 && id == 0 && tid == 0 && newCount) *newCount = n;
    if (id >= n) return;
    const Keypoint ok = oldKp[id];
    LkPoint pt;
    Keypoint *nk = pt.nk = &newKp[id];
    if (!ok.tracking_status) {
        if (tid == 0) {
            nk->x = ok.x; nk->y = ok.y; nk->strength = ok.strength; nk->tracking_status = ok.tracking_status;
            nk->scale = ok.scale; nk->error = ok.error;
        }
        return;
    }
    if (P.first + 1 == P.levels) {
        const float ptScale = P.level[P.first].ptScale;
        if (P.useEstimate) {
            const Keypoint ek = estKp[id];
            pt.x = (float)ek.x * ptScale;
            pt.y = (float)ek.y * ptScale;
            pt.status = ek.tracking_status;
            if (tid == 0) { nk->strength = ek.strength; nk->tracking_status = ek.tracking_status; nk->error = ek.error; }
        } else {
            pt.x = (float)ok.x * ptScale;
            pt.y = (float)ok.y * ptScale;
            pt.status = ok.tracking_status;
            if (tid == 0) { nk->tracking_status = ok.tracking_status; nk->strength = ok.strength; }
        }
    } else {
        const float2 q = next[id];
        pt.x = q.x * 2.0f;
        pt.y = q.y * 2.0f;
        pt.status = nk->tracking_status;
        __syncthreads();   // every lane has read next[id] and the status before lane 0 rewrites them
    }
    const int npix = (int)(P.winsz * P.winsz);
    int32_t *sI = lds, *sIx = sI + npix, *sIy = sIx + npix;
    float *sP0 = (float *)(sIy + npix), *sP1 = sP0 + npix, *sP2 = sP1 + npix, *sAcc = sP2 + npix;
    for (uint32_t lev = P.first;; lev--) {
        if (pt.status) lk_level<MAXW>(P, lev, ok, pt, sI, sIx, sIy, sP0, sP1, sP2, sAcc);
        if (lev == P.last) break;
        pt.x *= 2.0f;
        pt.y *= 2.0f;
        __syncthreads();   // the level's LDS is rewritten by the next
    }
    if (P.last != 0 && tid == 0) next[id] = make_float2(pt.x, pt.y);
}

struct LkLayout {
    size_t B, D, next, levels, base, total;   // `base` bytes suffice for the level-at-a-time form
};

inline LkLayout lk_layout(uint32_t w0, uint32_t h0, uint32_t capacity)
{
    LkLayout l;
    l.B = 0;
    l.D = align256(((size_t)2 * w0 + 64) * 2);
    l.next = align256(l.D + (size_t)w0 * h0 * 4);
    l.base = l.levels = align256(l.next + (size_t)capacity * 8);
    // derivative images of the levels above the finest: a third of it for halved levels, and their rounding
    l.total = align256(l.levels + (size_t)w0 * h0 * 4 / 2 + 16384);
    return l;
}

}  // namespace mvx

using namespace mvx;

extern "C" size_t mvx_OpticalFlowPyrLK_workspace_size(uint32_t width0, uint32_t height0, uint32_t capacity)
{
    return lk_layout(width0, height0, capacity ? capacity : 1).total;
}

extern "C" int mvx_OpticalFlowPyrLK_XY_XY(mvx_stream_t stream, void *pNewKeypoints, uint32_t *pNewCount,
                                          const mvx_image_level_t *oldPyramid, const mvx_image_level_t *newPyramid, uint32_t levels,
                                          float pyramidScale, const void *pOldKeypoints, const uint32_t *pOldCount,
                                          const void *pEstimates, uint32_t capacity, int32_t termination, float epsilon,
                                          uint32_t numIterations, int32_t useInitialEstimate, uint32_t windowDimension,
                                          void *workspace, size_t workspaceSize)
{
    if (!pNewKeypoints || !oldPyramid || !newPyramid || !pOldKeypoints || !pOldCount || !workspace || !capacity) return MVX_ERROR_INVALID_PARAMETERS;
    if (levels < 1 || levels > 16 || windowDimension < 3 || windowDimension > (uint32_t)LK_MAX_WIN) return MVX_ERROR_INVALID_PARAMETERS;
    if (useInitialEstimate && !pEstimates) return MVX_ERROR_INVALID_PARAMETERS;
    if ((uint32_t)termination != 0xF000u && (uint32_t)termination != TERM_EPSILON && (uint32_t)termination != TERM_BOTH)
        return MVX_ERROR_INVALID_PARAMETERS;
    const uint32_t w0 = oldPyramid[0].width, h0 = oldPyramid[0].height;
    for (uint32_t l = 0; l < levels; l++) {
        const mvx_image_level_t &o = oldPyramid[l], &nw = newPyramid[l];
        // the reference's Scharr loop needs 8 columns; the window must fit inside the level
        if (!o.ptr || !nw.ptr || o.width != nw.width || o.height != nw.height || o.width < 8 || o.height < 3 ||
            o.width > w0 || o.height > h0 || o.stride < o.width || nw.stride < nw.width)
            return MVX_ERROR_INVALID_PARAMETERS;
    }
    const LkLayout lay = lk_layout(w0, h0, capacity);
    if (workspaceSize < lay.base || ((uintptr_t)workspace & 15u)) return MVX_ERROR_INVALID_PARAMETERS;
    uint8_t *ws = (uint8_t *)workspace;
    uint16_t *B = (uint16_t *)(ws + lay.B) + 8;
    int16_t *D = (int16_t *)(ws + lay.D);
    float2 *next = (float2 *)(ws + lay.next);
    const hipStream_t st = stream_of(stream);
    LkParams P;
    P.levels = levels;
    P.winsz = windowDimension;
    P.halfWin = windowDimension >> 1;
    P.iterations = numIterations;
    P.termination = (uint32_t)termination;
    P.useEstimate = useInitialEstimate ? 1u : 0u;
    P.epsilon = epsilon;
    // one launch for all levels: a derivative image each, in the workspace's tail.  Levels may not grow upwards:
    // then a level's unwritten columns could hold a coarser level's values rather than the last call's.
    bool together = levels > 1;
    size_t at = lay.levels;
    for (uint32_t l = 0; l < levels; l++) {
        LkTrackLevel &t = P.level[l];
        t.img = LkLevel{oldPyramid[l].ptr, newPyramid[l].ptr, oldPyramid[l].width, oldPyramid[l].height, oldPyramid[l].stride, newPyramid[l].stride};
        t.ptScale = (float)pow((double)pyramidScale, (double)l);
        t.D = D;
        t.dStride = 2 * w0;
        if (l == 0) continue;
        t.D = (const int16_t *)(ws + at);
        t.dStride = 2 * t.img.width;
        at = align256(at + (size_t)t.img.width * t.img.height * 4);
        together = together && t.img.width <= P.level[l - 1].img.width && t.img.height <= P.level[l - 1].img.height;
    }
    together = together && at <= workspaceSize;
    const size_t ldsBytes = ((size_t)6 * windowDimension * windowDimension + 24) * 4;
    const auto track = [&](uint32_t first, uint32_t last) {
        P.first = first;
        P.last = last;
        hipLaunchKernelGGL(windowDimension <= (uint32_t)LK_SMALL_WIN ? k_lk_track<LK_SMALL_WIN> : k_lk_track<LK_MAX_WIN>, dim3(capacity), dim3(LK_THREADS), ldsBytes, st, P, next, (const Keypoint *)pOldKeypoints,
                           (const Keypoint *)pEstimates, (Keypoint *)pNewKeypoints, pOldCount, pNewCount, capacity);
    };
    for (int level = (int)levels - 1; level >= 0; level--) {
        LkTrackLevel &t = P.level[level];
        const bool own = together && level > 0;
        if (!own) { t.D = D; t.dStride = 2 * w0; }
        const uint32_t chunks = t.img.width / 8 + 1;   // one more for the columns past the last whole chunk
        hipLaunchKernelGGL(k_lk_scharr, dim3((chunks + 63) / 64, (t.img.height - 2 + 3) / 4), dim3(64, 4), 0, st, t.img, (int16_t *)t.D, t.dStride,
                           B, own ? (const int16_t *)D : nullptr, 2 * w0);
        if (!together) track((uint32_t)level, (uint32_t)level);
        MVX_LAUNCH_CHECK();
    }
    if (together) track(levels - 1, 0);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}
