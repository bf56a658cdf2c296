// canny.hip -- CannyEdgeDetector (gradient 3, 5, 7; L1 and L2 norms) for gfx950: Sobel -> non-max
// suppression with double threshold -> hysteresis.
//
// The reference traces hysteresis with a sequential LIFO stack on the CPU (its HIP backend has no
// trace kernel).  The traced image only depends on connectivity: a weak pixel ends at 255 iff it is
// 8-connected through weak pixels to a strong one.  Here that set is computed with a lock-free
// union-find over the edge pixels (atomicMin linking, then one find per pixel), three passes with no
// host round trip, in the 4-byte-per-pixel workspace the reference reserves for its XY stack.
#include "arith.hpp"
#include "rowmask.hpp"
#include <algorithm>

namespace mvx {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_dword __attribute__((aligned(4)));   // at a 4-byte aligned address
typedef uint32_t u32x2_dword __attribute__((ext_vector_type(2), aligned(4)));

inline bool plane_ok_c(const void *p, uint32_t w, uint32_t stride, uint32_t bpp)
{
    return p && aligned16(p) && (stride % 16u) == 0 && stride >= ((w * bpp + 15u) & ~15u);
}

// HafCpu_FastAtan2_Canny (ago_haf_cpu_arithmetic.cpp:9638-9656); statement order kept (0,0 -> 2)
MVX_DEV uint32_t canny_sector(int gx, int gy)
{
    const uint32_t ax = (uint32_t)abs(gx) & 0xffffu, ay = (uint32_t)abs(gy) & 0xffffu;
    const float d1 = (float)ax * 0.4142135623730950488016887242097f;
    const float d2 = (float)ax * 2.4142135623730950488016887242097f;
    uint32_t ret = (gx * gy) < 0 ? 3u : 1u;
    if ((float)ay <= d1) ret = 0;
    if ((float)ay >= d2) ret = 2;
    return ret;
}

// ---- Sobel planes, gradients 3, 5, 7, norms L1 and L2 (ago_haf_cpu_canny.cpp:44-427, 646-1056) -------------------
// 16-bit lane arithmetic of the reference's SSE code
MVX_DEV int w16(int v) { return (int16_t)(uint16_t)(uint32_t)v; }
MVX_DEV int s16(int v) { return min(max(v, -32768), 32767); }
MVX_DEV int sll16(int v, int k) { return w16((int)((uint32_t)(uint16_t)v << k)); }
MVX_DEV int abs16(int v) { return w16(v < 0 ? -v : v); }
MVX_DEV uint16_t canny_out(int mag16, uint32_t sector) { return (uint16_t)(sll16(mag16, 2) | (int)(sector & 3u)); }

// floor(sqrt(F)) for F < 2^32, exact: a float estimate corrected in integer arithmetic
MVX_DEV uint32_t isqrt_u64(uint64_t F)
{
    uint32_t k = (uint32_t)sqrtf((float)F);
    while ((uint64_t)k * k > F) k--;
    while ((uint64_t)(k + 1) * (k + 1) <= F) k++;
    return k;
}

// (vx_int16)sqrt((Gx*Gx) + (Gy*Gy)): 32-bit int sum, correctly rounded double sqrt truncated -- the
// integer square root -- with 0x80000000 for a negative (wrapped) sum, then 16 bits
MVX_DEV int l2_scalar(int gx, int gy)
{
    const int32_t q = (int32_t)((uint32_t)(gx * gx) + (uint32_t)(gy * gy));
    const int32_t t = q < 0 ? INT32_MIN : (int32_t)isqrt_u64((uint64_t)q);
    return (int16_t)(uint16_t)(uint32_t)t;
}

template <int G> struct Taps;
template <> struct Taps<3> { static constexpr int sm[3] = {1, 2, 1}, dv[3] = {-1, 0, 1}; };
template <> struct Taps<5> { static constexpr int sm[5] = {1, 4, 6, 4, 1}, dv[5] = {-1, -2, 0, 2, 1}; };
template <> struct Taps<7> { static constexpr int sm[7] = {1, 6, 15, 20, 15, 6, 1}, dv[7] = {-1, -4, -5, 0, 5, 4, 1}; };

// the scalar loop's value at (x, y), linear-address reads
template <int G, bool L2> MVX_DEV uint16_t canny_scalar(const uint8_t *src, long n, long stride, int x, int y)
{
    constexpr int R = G / 2;
    int gxs = 0, gys = 0;
#pragma unroll
    for (int j = 0; j < G; j++) {
        const long b = (long)(y - R + j) * stride + x;
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int p = (int)ld_u8(src, n, b + i - R);
            gxs += Taps<G>::sm[j] * Taps<G>::dv[i] * p;
            // 5x5 L2: the first row's term lacks its parentheses (ago_haf_cpu_canny.cpp:880)
            const int wy = (G == 5 && L2 && j == 0 && i > 0) ? Taps<G>::sm[i] : Taps<G>::dv[j] * Taps<G>::sm[i];
            gys += wy * p;
        }
    }
    const int gx = w16(gxs);
    int gy = w16(gys);
    if (G <= 5 && !L2) gy = w16(-gy);
    const int mag = L2 ? l2_scalar(gx, gy) : w16(abs(gx) + abs(gy));
    return canny_out(mag, canny_sector(gx, gy));
}

// The SSE passes over [0, aligned), aligned = w & ~15 >= 16: scratch rows r0, r1 (r1 = r0 + ALIGN16(w))
// with zeros before r0, after r1 and in their unwritten tails; a read past the end of r0 lands in r1
// (and one before r1 in r0) when w is a multiple of 16.  Each scratch slot x0-R .. stands for one source
// column (or none) for every row.  One wave owns a strip of 64 - 2R output columns and CSW_ROWS rows:
// lane l holds the slot of column x0 - R + l and keeps that column's G source bytes in a rolling
// registers (all of the strip's rows are loaded first); its two vertical sums reach the neighbouring lanes by DPP
// lane shifts, so no LDS and no barrier is involved.  Lanes R .. 63-R finish one column each; columns
// aligned-1 .. w-1 take the scalar loop's value.
// Only columns 0 .. 7 and those from aligned - 8 on need that (k_canny_sobel_g's edge waves); between them a
// window's slots are all in the row, and lanes own 8 columns (canny_columns).
constexpr int CSW_ROWS = 1;    // output rows per edge wave

// which scratch value a slot holds: kind 1 = (r0, r1) of source column sc, 2 = r0 <- r1 of sc (the slot
// lies past the end of r0), 3 = r1 <- r0 of sc (before the start of r1), 0 = zeros
MVX_DEV int canny_slot(int col, int aligned, int a16, int &sc)
{
    if (col >= 0 && col < aligned) { sc = col; return 1; }
    if (col >= a16 && col - a16 < aligned) { sc = col - a16; return 2; }
    if (col < 0 && a16 + col < aligned) { sc = a16 + col; return 3; }
    sc = 0;
    return 0;
}

// the vertical pass of the SSE loop over one column's G source bytes: t0 = the smoothing sum (scratch
// row r0), t1 = the derivative sum (r1); gradient 7 shifts both right by 2.  |t0| <= 4080 and
// |t1| <= 765 for every G, so the reference's 16-bit scratch values are these.
template <int G> MVX_DEV void canny_vsum(const int (&s)[G], int &t0, int &t1)
{
    if (G == 3) {
        t0 = s[0] + s[2] + 2 * s[1];
        t1 = s[2] - s[0];
    } else if (G == 5) {
        t0 = 4 * (s[1] + s[3]) + 6 * s[2] + (s[0] + s[4]);
        t1 = 2 * (s[3] - s[1]) + (s[4] - s[0]);
    } else {
        t0 = (6 * (s[1] + s[5]) + 20 * s[3] + (s[0] + s[6]) + 15 * (s[2] + s[4])) >> 2;
        t1 = (4 * (s[5] - s[1]) + (s[6] - s[0]) + 5 * (s[4] - s[2])) >> 2;
    }
}

// the value of lane + 1 / lane - 1 (DPP wave_shl:1 / wave_shr:1; lanes past the ends read 0)
MVX_DEV int dpp_next(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
MVX_DEV int dpp_prev(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }

// the SSE horizontal pass and packing of one column from the scratch slots at offsets -R..R
// (A0(d) = r0 slot, A1(d) = r1 slot)
template <int G, bool L2> MVX_DEV uint16_t canny_simd_px(const int (&a0)[G], const int (&a1)[G])
{
    constexpr int R = G / 2;
#define A0(d) (a0[R + (d)])
#define A1(d) (a1[R + (d)])
    int gx, gy;
    if (G == 3) {
        gx = w16(A0(1) - A0(-1));
        gy = w16(-w16(w16(A1(-1) + A1(1)) + sll16(A1(0), 1)));
    } else if (G == 5) {
        gx = s16(sll16(w16(A0(1) - A0(-1)), 1) + w16(A0(2) - A0(-2)));
        int t = w16(sll16(w16(A1(-1) + A1(1)), 2) + w16(A1(-2) + A1(2)));
        t = L2 ? s16(t + w16(A1(0) * 6)) : w16(t + w16(A1(0) * 6));
        gy = w16(-t);
    } else {
        int t = sll16(s16(A0(2) - A0(-2)), 2);
        const int u = w16(s16(A0(1) - A0(-1)) * 5);
        t = s16(t + s16(A0(3) - A0(-3)));
        gx = s16(t + u);
        int v = s16(w16(w16(A1(-2) + A1(2)) * 6) + w16(A1(0) * 20));
        const int q = w16(w16(A1(-1) + A1(1)) * 15);
        v = s16(v + s16(A1(-3) + A1(3)));
        v = s16(v + q);
        gy = s16(-v);
    }
#undef A0
#undef A1
    int mag;
    if (!L2) {
        mag = w16(abs16(gx) + abs16(gy));
        if (G == 7 && mag > 0x3fff) mag = 0x3fff;
    } else if (G == 3) {
        mag = l2_pack_simd((float)(uint16_t)w16(gx * gx) + (float)(uint16_t)w16(gy * gy));
    } else {
        mag = l2_pack_simd((float)(gx * gx + gy * gy));
    }
    return canny_out(mag, canny_sector(gx, gy));
}

// one strip: output columns xs .. xe - 1 (at most 64 - 2R), rows yb .. ye - 1
template <int G, bool L2>
MVX_DEV void canny_strip(uint32_t w, uint32_t h, uint16_t *dst, uint32_t dstStride, const uint8_t *src, uint32_t srcStride,
                         int xs, int xe, int yb, int ye)
{
    constexpr int R = G / 2;
    const int lane = (int)threadIdx.x & 63;
    const int aligned = (int)(w & ~15u), a16 = (int)((w + 15u) & ~15u);
    const int col = xs - R + lane;
    int sc = col;
    const int kind = canny_slot(col, aligned, a16, sc);
    gptr_t<const uint8_t> sp = gmem(src);
    gptr_t<uint8_t> dp = (gptr_t<uint8_t>)gmem(dst);
    // a zero slot still loads an in-plane byte (column 0) and drops it, so the loads stay unconditional
    auto load = [&](int r) -> int {
        const int v = sp[(uint64_t)(uint32_t)r * srcStride + (uint32_t)sc];
        return kind == 0 ? 0 : v;
    };
    // every source row of the strip is loaded before the first is used: the loads are all in flight
    // together, and row i waits only for its own G rows
    constexpr int NR = CSW_ROWS + G - 1;
    int rw[NR];
#pragma unroll
    for (int j = 0; j < NR; j++) rw[j] = (yb - R + j < ye + R) ? load(yb - R + j) : 0;
    const int x = col;   // output column of lanes R .. 63 - R
    const bool outLane = lane >= R && lane < 64 - R && x < xe;
#pragma unroll
    for (int i = 0; i < CSW_ROWS; i++) {
        const int y = yb + i;
        if (y >= ye) break;
        int win[G];
#pragma unroll
        for (int j = 0; j < G; j++) win[j] = rw[i + j];
        int t0, t1;
        canny_vsum<G>(win, t0, t1);
        int a0[G], a1[G];
        a0[R] = kind == 1 ? t0 : kind == 2 ? t1 : 0;
        a1[R] = kind == 1 ? t1 : kind == 3 ? t0 : 0;
        // the lane shifts run with every lane active
#pragma unroll
        for (int d = 1; d <= R; d++) {
            a0[R + d] = dpp_next(a0[R + d - 1]);
            a0[R - d] = dpp_prev(a0[R - d + 1]);
            a1[R + d] = dpp_next(a1[R + d - 1]);
            a1[R - d] = dpp_prev(a1[R - d + 1]);
        }
        uint16_t out = canny_simd_px<G, L2>(a0, a1);
        if (outLane) {
            if (x >= aligned - 1) out = canny_scalar<G, L2>(src, (long)h * srcStride, srcStride, x, y);
            *(gptr_t<uint16_t>)(dp + (uint64_t)(uint32_t)y * dstStride + 2 * (uint32_t)x) = out;
        }
    }
}

// Eight columns of a lane: x0 .. x0+7 with 8 <= x0 and x0 + 16 <= aligned, CSC_ROWS rows down.  A lane loads the
// 16 bytes from x0 - 4 on of each row, so that no lane waits for another; sums are pairs of 16-bit columns, the
// even ones of four columns k and the odd ones (E_k, O_k), and the pairs one or two columns on are shifts by half
// a register.  Every sum but the gradient-7 ones' last is exact in 16 bits, that one saturates as the SSE code's
// does; the rest of a pixel is a few float operations.
typedef short i16x2 __attribute__((ext_vector_type(2)));

MVX_DEV i16x2 i16_pair(uint32_t v) { return __builtin_bit_cast(i16x2, v); }
MVX_DEV uint32_t bits_of(i16x2 v) { return __builtin_bit_cast(uint32_t, v); }
MVX_DEV i16x2 pair_shift(i16x2 a, i16x2 b) { return i16_pair(__builtin_amdgcn_alignbit(bits_of(b), bits_of(a), 16)); }
MVX_DEV i16x2 pair_abs(i16x2 v) { return __builtin_elementwise_max(v, (i16x2)(0 - v)); }

// pairs of 2 and of 4 that the compiler cannot see through: it would split a multiply-add by them into a shift
// and an add, two instructions for one
struct CannyMul { i16x2 two, four; };
MVX_DEV CannyMul canny_mul()
{
    uint32_t two = 0x00020002u, four = 0x00040004u;
    asm("" : "+s"(two), "+s"(four));
    return {i16_pair(two), i16_pair(four)};
}

// canny_vsum for two columns
template <int G> MVX_DEV void canny_vsum2(const i16x2 (&s)[G], const CannyMul &k, i16x2 &t0, i16x2 &t1)
{
    if constexpr (G == 3) {
        t0 = s[1] * k.two + (s[0] + s[2]);
        t1 = s[2] - s[0];
    } else if constexpr (G == 5) {
        t0 = s[2] * (short)6 + ((s[1] + s[3]) * k.four + (s[0] + s[4]));
        t1 = (s[3] - s[1]) * k.two + (s[4] - s[0]);
    } else {
        t0 = ((s[0] + s[G - 1]) + (s[1] + s[G - 2]) * (short)6 + (s[2] + s[G - 3]) * (short)15 + s[G / 2] * (short)20) >> (short)2;
        t1 = ((s[G - 1] - s[0]) + (s[G - 2] - s[1]) * k.four + (s[G - 3] - s[2]) * (short)5) >> (short)2;
    }
}

// the gradients of a pair of columns from the pairs at columns -R .. R of it (canny_simd_px's, gy's sign included)
template <int G> MVX_DEV void canny_grad2(const i16x2 (&a0)[G], const i16x2 (&a1)[G], const CannyMul &k, i16x2 &gx, i16x2 &gy)
{
    if constexpr (G == 3) {
        gx = a0[2] - a0[0];
        gy = (short)0 - (a1[1] * k.two + (a1[0] + a1[2]));
    } else if constexpr (G == 5) {
        gx = (a0[3] - a0[1]) * k.two + (a0[4] - a0[0]);
        gy = (short)0 - (a1[2] * (short)6 + ((a1[1] + a1[3]) * k.four + (a1[0] + a1[4])));
    } else {
        gx = __builtin_elementwise_add_sat((i16x2)((a0[G - 2] - a0[1]) * k.four + (a0[G - 1] - a0[0])),
                                           (i16x2)((a0[G - 3] - a0[2]) * (short)5));
        const i16x2 v = __builtin_elementwise_add_sat((i16x2)((a1[1] + a1[G - 2]) * (short)6 + a1[G / 2] * (short)20 + (a1[0] + a1[G - 1])),
                                                      (i16x2)((a1[2] + a1[G - 3]) * (short)15));
        gy = __builtin_elementwise_sub_sat((i16x2)(short)0, v);
    }
}

// a pixel's sector (canny_sector) given 3 or 1 for gx * gy negative or not
MVX_DEV uint32_t canny_sector_f(float fx, float fy, uint32_t diagonal)
{
    uint32_t ret = fabsf(fy) <= fabsf(fx) * 0.4142135623730950488016887242097f ? 0u : diagonal;
    return fabsf(fy) >= fabsf(fx) * 2.4142135623730950488016887242097f ? 2u : ret;
}

template <int G, bool L2> MVX_DEV uint32_t canny_pair(i16x2 gx, i16x2 gy)
{
    // where one of the two is zero the sector is 0 or 2 whatever the signs
    const uint32_t diag = (((bits_of(gx) ^ bits_of(gy)) >> 14) & 0x00020002u) | 0x00010001u;
    const uint32_t sec = canny_sector_f((float)gx.x, (float)gy.x, diag & 0xffffu) | (canny_sector_f((float)gx.y, (float)gy.y, diag >> 16) << 16);
    uint32_t mag;
    if (L2) {
        uint32_t m0, m1;
        if (G == 3) {   // the squares wrap at 16 bits
            const u16x2 xx = pair_of(bits_of(gx)) * pair_of(bits_of(gx)), yy = pair_of(bits_of(gy)) * pair_of(bits_of(gy));
            m0 = l2_round((float)xx.x + (float)yy.x);
            m1 = l2_round((float)xx.y + (float)yy.y);
        } else {
            const i16x2 p0 = i16_pair(__builtin_amdgcn_perm(bits_of(gy), bits_of(gx), 0x05040100u));
            const i16x2 p1 = i16_pair(__builtin_amdgcn_perm(bits_of(gy), bits_of(gx), 0x07060302u));
            m0 = l2_round((float)__builtin_amdgcn_sdot2(p0, p0, 0, false));
            m1 = l2_round((float)__builtin_amdgcn_sdot2(p1, p1, 0, false));
        }
        mag = __builtin_amdgcn_perm(m1, m0, 0x05040100u);   // at most 46341: no saturation
    } else {
        i16x2 m = pair_abs(gx) + pair_abs(gy);
        if (G == 7) m = __builtin_elementwise_min(m, (i16x2)(short)0x3fff);
        mag = bits_of(m);
    }
    return bits_of((u16x2)(pair_of(mag) << (unsigned short)2)) | sec;
}

constexpr int CSC_ROWS = 4;    // output rows per lane

template <int G, bool L2>
MVX_DEV void canny_columns(uint32_t h, uint16_t *dst, uint32_t dstStride, const uint8_t *src, uint32_t srcStride, uint32_t x0, uint32_t rowGroup)
{
    constexpr int R = G / 2;
    const int yb = R + (int)rowGroup * CSC_ROWS, last = (int)h - 1;
    gptr_t<const uint8_t> p = gmem(src) + (x0 - 4);
    u32x4 raw[CSC_ROWS + 2 * R];
#pragma unroll
    for (int j = 0; j < CSC_ROWS + 2 * R; j++) raw[j] = *(gptr_t<const u32x4_dword>)(p + (uint64_t)(uint32_t)min(yb - R + j, last) * srcStride);
    // here all rows have arrived: left alone the compiler moves some of the loads down to their first use
#pragma unroll
    for (int j = 0; j < CSC_ROWS + 2 * R; j++) asm volatile("" : "+v"(raw[j]));
    const CannyMul mul = canny_mul();
    i16x2 win[G][8];   // the rows' columns: [2k] = E_k, [2k + 1] = O_k
#pragma unroll
    for (int j = 0; j < CSC_ROWS + 2 * R; j++) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            win[j % G][2 * k] = i16_pair(bits_of(even_bytes(raw[j][k])));
            win[j % G][2 * k + 1] = i16_pair(bits_of(odd_bytes(raw[j][k])));
        }
        if (j < 2 * R) continue;
        const int y = yb + j - 2 * R;
        i16x2 t0[8], t1[8];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            i16x2 s[G];
#pragma unroll
            for (int i = 0; i < G; i++) s[i] = win[(j + 1 + i) % G][c];   // oldest first
            canny_vsum2<G>(s, mul, t0[c], t1[c]);
        }
        uint32_t out[4];
#pragma unroll
        for (int c = 2; c < 6; c++) {   // E_1, O_1, E_2, O_2
            // the pair d columns on of E_k (c even) or O_k: O_k's columns are one on from E_k's
            const auto at = [&](const i16x2 (&t)[8], int d) -> i16x2 {
                const int n = (c & 1) + d, k = c / 2;       // columns from E_k
                const int q = n & 1, m = (n - q) / 2;       // pair kind (even or odd), half pairs on
                const int i = 2 * (k + (m - (m & 1)) / 2) + q;
                return (m & 1) ? pair_shift(t[i], t[i + 2]) : t[i];
            };
            i16x2 a0[G], a1[G];
#pragma unroll
            for (int d = -R; d <= R; d++) {
                a0[R + d] = at(t0, d);
                a1[R + d] = at(t1, d);
            }
            i16x2 gx, gy;
            canny_grad2<G>(a0, a1, mul, gx, gy);
            out[c - 2] = canny_pair<G, L2>(gx, gy);
        }
        u32x4 o;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            o[2 * k] = __builtin_amdgcn_perm(out[2 * k + 1], out[2 * k], 0x05040100u);
            o[2 * k + 1] = __builtin_amdgcn_perm(out[2 * k + 1], out[2 * k], 0x07060302u);
        }
        // the rows past the last are computed and dropped: a branch around them would hold their loads back
        if (y <= last - R) *(gptr_t<u32x4>)((gptr_t<uint8_t>)gmem(dst) + (uint64_t)(uint32_t)y * dstStride + 2 * x0) = o;
    }
}

// The first `edge` workgroups' waves take the left and right edge of CSW_ROWS rows each (first, since theirs are the
// longest chains); the others 8-column units of the columns between, row group after row group.
// 3840x2160, gradient 5, L2: 30.5 us with a lane a column and shifts between lanes (83 lane operations a pixel), 18.0 now
// (41): half of it vector instructions, the rest the waits for memory at either end of four rows.
template <int G, bool L2>
__global__ void __launch_bounds__(256)
k_canny_sobel_g(uint32_t w, uint32_t h, uint16_t *__restrict__ dst, uint32_t dstStride, const uint8_t *__restrict__ src,
                uint32_t srcStride, uint32_t edge, uint32_t units, uint32_t rowGroups)
{
    constexpr int R = G / 2;
    const uint32_t aligned = w & ~15u;
    if (blockIdx.x >= edge) {
        const uint32_t u = (blockIdx.x - edge) * 256 + threadIdx.x, g = u / units;
        if (g < rowGroups) canny_columns<G, L2>(h, dst, dstStride, src, srcStride, 8 + 8 * (u - g * units), g);
        return;
    }
    const int e = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int yb = R + (e >> 1) * CSW_ROWS, ye = min(yb + CSW_ROWS, (int)h - R);
    if (yb >= ye) return;
    if (e & 1) canny_strip<G, L2>(w, h, dst, dstStride, src, srcStride, (int)aligned - 8, (int)w, yb, ye);
    else canny_strip<G, L2>(w, h, dst, dstStride, src, srcStride, 0, 8, yb, ye);
}

// widths below 16: only the scalar loop runs, from x = -1 (the slot before each row), rows in order
template <int G, bool L2>
__global__ void k_canny_sobel_g_narrow(uint32_t w, uint32_t h, uint16_t *dst, uint32_t dstStride, const uint8_t *src,
                                       uint32_t srcStride)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    constexpr int R = G / 2;
    const long n = (long)h * srcStride;
    for (int y = R; y < (int)h - R; y++)
        for (int x = -1; x < (int)w; x++)
            *(uint16_t *)((uint8_t *)dst + (long)y * dstStride + 2L * x) = canny_scalar<G, L2>(src, n, srcStride, x, y);
}

// CannySuppThreshold_U8XY_U16_3x3 (ago_haf_cpu_canny.cpp:549-596): x in [1, w-2], y in [1, h-2].
// A lane owns 8 columns and SUP_ROWS rows; it loads each row's 16 bytes and the words beside them, all rows first.
// Pixels run two to a register: the larger neighbour along each of the four directions, the one of the pixel's
// sector picked by its two bits, comparisons as saturating differences clamped to 1.
// Bound by memory (3 bytes a pixel) and latency.  3840x2160: rows staged in LDS a dword a value 11.6 us, 10.8 now.
constexpr int SUP_ROWS = 4;

// a > b: 1, else 0
MVX_DEV u16x2 pair_above(u16x2 a, u16x2 b, u16x2 one) { return __builtin_elementwise_min(__builtin_elementwise_sub_sat(a, b), one); }

// lowerP and upperP: the thresholds plus 1, clamped to 0 .. 16384 (a suppressed pixel's value plus 1 is 1 .. 16384)
__global__ void __launch_bounds__(256)
k_canny_supp(uint32_t w, uint32_t h, uint8_t *__restrict__ dst, uint32_t dstStride, const uint16_t *__restrict__ mag,
             uint32_t magStride, uint32_t lowerP, uint32_t upperP, uint32_t units, uint32_t rowGroups)
{
    const uint32_t u = blockIdx.x * 256 + threadIdx.x, g = u / units;
    if (g >= rowGroups) return;
    const uint32_t x0 = 8 * (u - g * units);
    const int yb = 1 + (int)g * SUP_ROWS, last = (int)h - 1;
    // the 16-byte chunk that starts inside the row lies inside its ALIGN16 bytes, which the stride covers; the words
    // beside it are only read where an output needs them
    const uint32_t lo = x0 ? x0 - 2 : 0u, hi = x0 + 8 < w ? x0 + 8 : x0;
    gptr_t<const uint8_t> p = gmem((const uint8_t *)mag);
    uint32_t raw[SUP_ROWS + 2][6];
#pragma unroll
    for (int j = 0; j < SUP_ROWS + 2; j++) {
        gptr_t<const uint8_t> r = p + (uint64_t)(uint32_t)min(yb - 1 + j, last) * magStride;
        const u32x4 v = *(gptr_t<const u32x4>)(r + 2 * x0);
        raw[j][0] = *(gptr_t<const uint32_t>)(r + 2 * lo);
        raw[j][5] = *(gptr_t<const uint32_t>)(r + 2 * hi);
#pragma unroll
        for (int k = 0; k < 4; k++) raw[j][1 + k] = v[k];
    }
    // here all rows have arrived: left alone the compiler moves some of the loads down to their first use
#pragma unroll
    for (int j = 0; j < SUP_ROWS + 2; j++)
#pragma unroll
        for (int k = 0; k < 6; k++) asm volatile("" : "+v"(raw[j][k]));
    uint32_t oneBits = 0x00010001u;   // not known to the compiler, which would turn the comparisons into one per half
    asm("" : "+s"(oneBits));
    const u16x2 one = pair_of(oneBits);
    const u16x2 lower = pair_of(lowerP | (lowerP << 16)), upper = pair_of(upperP | (upperP << 16));
    u16x2 m[3][6], n[3][5];   // magnitudes of three rows: column pairs x0-2 .. x0+9, and those one column on
#pragma unroll
    for (int j = 0; j < SUP_ROWS + 2; j++) {
#pragma unroll
        for (int k = 0; k < 6; k++) m[j % 3][k] = pair_of(raw[j][k]) >> (unsigned short)2;
#pragma unroll
        for (int k = 0; k < 5; k++) n[j % 3][k] = pair_shift(m[j % 3][k], m[j % 3][k + 1]);
        if (j < 2) continue;
        const int a = (j + 1) % 3, b = (j + 2) % 3, c = j % 3;   // rows y - 1, y, y + 1
        const int y = yb + j - 2;
        uint32_t out[4];
#pragma unroll
        for (int k = 1; k < 5; k++) {
            // neighbour pairs by sector (ago_haf_cpu_canny.cpp:26-31): 0 (-1,0)/(1,0), 1 (1,-1)/(-1,1),
            // 2 (0,-1)/(0,1), 3 (-1,-1)/(1,1)
            const u16x2 d0 = __builtin_elementwise_max(n[b][k - 1], n[b][k]), d1 = __builtin_elementwise_max(n[a][k], n[c][k - 1]);
            const u16x2 d2 = __builtin_elementwise_max(m[a][k], m[c][k]), d3 = __builtin_elementwise_max(n[a][k - 1], n[c][k]);
            const u16x2 v = pair_of(raw[j - 1][k]);
            const uint32_t s0 = bits_of((u16x2)(u16x2(0) - (v & one)));
            const uint32_t s1 = bits_of((u16x2)(u16x2(0) - ((v >> (unsigned short)1) & one)));
            const uint32_t e = (s0 & bits_of(d1)) | (~s0 & bits_of(d0)), o = (s0 & bits_of(d3)) | (~s0 & bits_of(d2));
            const u16x2 d = pair_of((s1 & o) | (~s1 & e));
            const u16x2 edge = m[b][k] * pair_above(m[b][k], d, one) + one;
            out[k - 1] = bits_of((u16x2)(pair_above(edge, lower, one) * (unsigned short)127 + (pair_above(edge, upper, one) << (unsigned short)7)));
        }
        if (y >= last) continue;
        const uint32_t b0 = __builtin_amdgcn_perm(out[1], out[0], 0x06040200u), b1 = __builtin_amdgcn_perm(out[3], out[2], 0x06040200u);
        gptr_t<uint8_t> q = gmem(dst) + (uint64_t)(uint32_t)y * dstStride + x0;
        if (x0 >= 1 && x0 + 8 <= w - 1) {
            *(gptr_t<u32x2_dword>)q = u32x2_dword{b0, b1};
        } else {
            for (uint32_t i = x0 ? 0u : 1u; i < 8 && x0 + i + 2 <= w; i++) q[i] = (uint8_t)((i < 4 ? b0 : b1) >> (8 * (i & 3)));
        }
    }
}

// seed the union-find: every interior edge pixel (127 or 255) is its own root.  Labels always point
// to a smaller or equal index of an edge pixel, so finds terminate whatever the image holds.
__global__ void __launch_bounds__(256)
k_canny_init(uint32_t w, uint32_t h, const uint8_t *__restrict__ img, uint32_t stride, uint32_t *__restrict__ lab)
{
    const int x = 1 + (int)(blockIdx.x * 256 + threadIdx.x);
    const int y = 1 + (int)blockIdx.y;
    if (x >= (int)w - 1 || y >= (int)h - 1) return;
    if (img[(long)y * stride + x]) lab[(long)y * w + x] = (uint32_t)((long)y * w + x);
}

MVX_DEV uint32_t uf_find(const uint32_t *lab, uint32_t p)
{
    uint32_t l = lab[p] & 0x7fffffffu;
    while (l != p) {
        p = l;
        l = lab[p] & 0x7fffffffu;
    }
    return p;
}

// link the trees of a and b: the larger root points at the smaller (atomicMin), retried until the
// roots agree; lock-free and order independent
MVX_DEV void uf_union(uint32_t *lab, uint32_t a, uint32_t b)
{
    while (true) {
        a = uf_find(lab, a);
        b = uf_find(lab, b);
        if (a == b) return;
        if (a < b) { uint32_t t = a; a = b; b = t; }   // a > b: hang a under b
        const uint32_t old = atomicMin(&lab[a], b);
        if (old == a) return;
        a = old;
    }
}

// merge each edge pixel with its E, SW, S, SE edge neighbours (covers all 8-neighbour pairs)
__global__ void __launch_bounds__(256)
k_canny_merge(uint32_t w, uint32_t h, const uint8_t *__restrict__ img, uint32_t stride, uint32_t *__restrict__ lab)
{
    const int x = 1 + (int)(blockIdx.x * 256 + threadIdx.x);
    const int y = 1 + (int)blockIdx.y;
    if (x >= (int)w - 1 || y >= (int)h - 1) return;
    const uint8_t *r0 = img + (long)y * stride;
    if (!r0[x]) return;
    const uint8_t *r1 = r0 + stride;
    const uint32_t p = (uint32_t)((long)y * w + x);
    // only interior neighbours carry labels (the border rows/columns are outside the supp range)
    const bool right = x + 1 < (int)w - 1, below = y + 1 < (int)h - 1, left = x - 1 >= 1;
    if (right && r0[x + 1]) uf_union(lab, p, p + 1);
    if (below && left && r1[x - 1]) uf_union(lab, p, p + w - 1);
    if (below && r1[x]) uf_union(lab, p, p + w);
    if (below && right && r1[x + 1]) uf_union(lab, p, p + w + 1);
}

__global__ void __launch_bounds__(256)
k_canny_mark(uint32_t w, uint32_t h, const uint8_t *__restrict__ img, uint32_t stride, uint32_t *__restrict__ lab)
{
    const int x = 1 + (int)(blockIdx.x * 256 + threadIdx.x);
    const int y = 1 + (int)blockIdx.y;
    if (x >= (int)w - 1 || y >= (int)h - 1) return;
    if (img[(long)y * stride + x] != 255) return;
    const uint32_t r = uf_find(lab, (uint32_t)((long)y * w + x));
    atomicOr(&lab[r], 0x80000000u);
}

__global__ void __launch_bounds__(256)
k_canny_final(uint32_t w, uint32_t h, uint8_t *__restrict__ img, uint32_t stride, const uint32_t *__restrict__ lab)
{
    const int x = 1 + (int)(blockIdx.x * 256 + threadIdx.x);
    const int y = 1 + (int)blockIdx.y;
    if (x >= (int)w - 1 || y >= (int)h - 1) return;
    uint8_t *p = img + (long)y * stride + x;
    if (*p != 127) return;
    const uint32_t r = uf_find(lab, (uint32_t)((long)y * w + x));
    *p = (lab[r] & 0x80000000u) ? 255 : 0;
}

// ---------------------------------------------------------------- tiled edge trace ----------------
// HafCpu_CannyEdgeTrace_U8_U8XY (ago_haf_cpu_canny.cpp:598-645): every 127 pixel 8-connected to a 255
// pixel through 127 pixels becomes 255, every other 127 becomes 0.  The image is cut into 64x16 tiles; the
// edge (127 or 255) and strong (255) pixels of a tile's interior become 64-bit row masks.  Two dilations
// inside the tile, one from the strong pixels, one from the tile-border edge pixels it did not reach: pixels
// the first reaches are final 255; edge pixels reached by neither are final 0; the rest (components that
// touch the tile border and hold no strong pixel) stay 127 and get a union-find id, the k-th such component
// of tile t the id 1 + t*CT_NB + k (at most one per border pixel).  Border tables record per border pixel
// CT_NONE, 0 (the strong node) or 1 + k, seed tables one pixel of each component.  A second pass unions
// the tables across tile edges, a third grows the components whose root is the strong node from their
// seeds and writes 255 there and 0 at the tile's other 127 pixels.
//
// One wave takes four tiles side by side, lane = tile * 16 + row: a row's 64 pixels are four 16-byte loads of
// its lane, their masks come from byte-wise arithmetic and dot products with powers of two (9 operations per
// 4 pixels), the lanes above and below are DPP shifts inside 16 lanes, and all four tiles grow, and find
// their k-th component, together.  A wave per tile with a lane per column spent 1285 vector instructions a
// tile on per-row ballots, per-row stores and 16 busy lanes of 64 (3840x2160, 3% edge pixels: tile pass
// 24.7 us, resolve pass 14.2 us; now 13.1 and 5.3).
constexpr int CT_W = 64, CT_H = 16, CT_NB = 2 * (CT_W + CT_H), CT_QUAD = 4;
constexpr uint32_t CT_NONE = 0xffffu;

struct CtArgs {
    uint32_t w, h, stride, tilesX, tilesY, quadsX;
    uint8_t *img;
    uint32_t *parent;   // 1 + tiles * CT_NB: slot 0 the strong node (its own root), then CT_NB per tile
    uint16_t *border;   // tiles * 2 * CT_NB: top row, bottom row (CT_W each), left, right column (CT_H each), seeds (CT_NB)
    uint32_t *ucount;   // tiles: undecided components of the tile
};

// a lane's row of its tile; lanes past the image hold no pixel
struct CtRow {
    int lane, row, tile, tx0, tw, th, ty0;
    bool in;          // the lane's tile is in the image
    uint64_t inner;   // the row's pixels in the image's interior
    u32x4 x[4];       // its 64 bytes; junk where outside the image
};

MVX_DEV bool ct_row(const CtArgs &a, CtRow &t)
{
    const uint32_t q = blockIdx.x * 4 + (uint32_t)__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (q >= a.quadsX * a.tilesY) return false;
    t.lane = (int)threadIdx.x & 63;
    t.row = t.lane & 15;
    const int tY = (int)(q / a.quadsX), tX = (int)(q % a.quadsX) * CT_QUAD + (t.lane >> 4);
    t.in = tX < (int)a.tilesX;
    t.tile = tY * (int)a.tilesX + tX;
    t.tx0 = tX * CT_W;
    t.ty0 = tY * CT_H;
    t.tw = min(CT_W, (int)a.w - t.tx0);
    t.th = min(CT_H, (int)a.h - t.ty0);
    const int y = t.ty0 + t.row, n = (int)a.w - 1 - t.tx0;   // columns below n are left of the image's last
    uint64_t cols = n >= CT_W ? ~0ull : n > 0 ? (1ull << n) - 1 : 0ull;
    if (tX == 0) cols &= ~1ull;
    t.inner = (y >= 1 && y <= (int)a.h - 2) ? cols : 0ull;
    return true;
}

// a 16-byte chunk that starts left of column w lies inside the row's ALIGN16(w) bytes, which the stride covers
MVX_DEV void ct_load(const CtArgs &a, CtRow &t)
{
    gptr_t<const uint8_t> p = gmem((const uint8_t *)a.img) + (long)(t.ty0 + t.row) * a.stride + t.tx0;
    const int n = t.inner ? t.tw : 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        t.x[c] = u32x4{0u, 0u, 0u, 0u};
        if (16 * c < n) t.x[c] = *(gptr_t<const u32x4>)(p + 16 * c);
    }
}

// bit i: byte i of the row is 127 or 255 (edge), 255 (strong).  With z = byte ^ 127, an edge's low seven bits
// are zero and adding 127 leaves bit 7 clear; a dot product with 1, 2, 4 .. 128 collects eight bytes' bits.
MVX_DEV void ct_masks(const CtRow &t, uint64_t &edge, uint64_t &strong)
{
    uint32_t eb[2] = {0u, 0u}, sb[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; i++) {   // eight columns
        uint32_t ae = 0, as = 0;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t z = t.x[i / 2][2 * (i % 2) + j] ^ 0x7f7f7f7fu;
            const uint32_t e = ~((z & 0x7f7f7f7fu) + 0x7f7f7f7fu) & 0x80808080u, s = e & z;
            const uint32_t weights = j ? 0x80402010u : 0x08040201u;
            ae = __builtin_amdgcn_udot4(e, weights, ae, false);
            as = __builtin_amdgcn_udot4(s, weights, as, false);
        }
        const int at = 8 * (i % 4) - 7;   // the sums are 128 times the byte of bits
        eb[i / 4] |= at < 0 ? ae >> 7 : ae << (at < 0 ? 0 : at);
        sb[i / 4] |= at < 0 ? as >> 7 : as << (at < 0 ? 0 : at);
    }
    edge = (((uint64_t)eb[1] << 32) | eb[0]) & t.inner;
    strong = (((uint64_t)sb[1] << 32) | sb[0]) & t.inner;
}

// four bits -> four bytes of 0 or 255
MVX_DEV uint32_t ct_bytes(uint32_t nibble)
{
    const uint32_t v = __umul24(nibble, 0x00204081u) & 0x01010101u;
    return (v << 8) - v;
}

// the row's pixels in `set` become 255 where `on`, else 0.  Chunks that hold one are stored whole, except that
// nothing at or past column w is written.
MVX_DEV void ct_store(const CtArgs &a, const CtRow &t, uint64_t set, uint64_t on)
{
    gptr_t<uint8_t> p = gmem(a.img) + (long)(t.ty0 + t.row) * a.stride + t.tx0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t s = (uint32_t)(set >> (16 * c)) & 0xffffu, o = (uint32_t)(on >> (16 * c)) & 0xffffu;
        if (s == 0) continue;
        u32x4 v;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t m = ct_bytes((s >> (4 * j)) & 15u);
            v[j] = (t.x[c][j] & ~m) | (ct_bytes((o >> (4 * j)) & 15u) & m);
        }
        if (16 * c + 16 <= t.tw) {
            *(gptr_t<u32x4>)(p + 16 * c) = v;
        } else {
            for (uint32_t left = s; left; left &= left - 1) {
                const int i = __builtin_ctz(left);
                p[16 * c + i] = (o >> i) & 1u ? 255 : 0;
            }
        }
    }
}

template <int CTRL> MVX_DEV uint64_t ct_dpp64(uint64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, true);
    return ((uint64_t)hi << 32) | lo;
}

// The runs of set bits of e that hold a bit of m (m inside e), from each such bit upwards: adding m to e carries
// through a run from its lowest bit of m on, and where the sum's bit is clear the carry passed over a bit of e.
MVX_DEV uint64_t fill_up(uint64_t m, uint64_t e)
{
    const uint64_t t = e + m;
    return (t & m) | (~t & e);
}

// Grow m (inside e) by 8-connectivity until nothing changes, in each 16 lanes on their own.  A round fills whole
// runs of a row by carries and steps one row up and down (row_shr:1 and row_shl:1, zeros past the 16 lanes), so
// the rounds are as many as the rows that a component winds through.  Called by the whole wave.
MVX_DEV uint64_t ct_grow(uint64_t m, uint64_t e)
{
    const uint64_t er = __builtin_bitreverse64(e);
    while (true) {
        const uint64_t f = __builtin_bitreverse64(fill_up(__builtin_bitreverse64(fill_up(m, e)), er));
        uint64_t v = ct_dpp64<0x111>(f) | ct_dpp64<0x101>(f);
        v |= (v << 1) | (v >> 1);
        m = (v & e) | f;
        if (!__any(m != f)) return m;
    }
}

// The border codes of four columns (lane j of a tile: columns 4j .. 4j+3) of one row, two 16-bit codes a word:
// where the row's mask has a bit the code becomes `code`.
MVX_DEV void ct_codes(uint32_t (&v)[2], uint64_t rowMask, int row, uint32_t code)
{
    const uint32_t n = (uint32_t)(rowMask >> (4 * row));
    const uint32_t both = code | (code << 16);
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t b0 = 0u - ((n >> (2 * j)) & 1u), b1 = 0u - ((n >> (2 * j + 1)) & 1u);
        const uint32_t m = (b0 & 0xffffu) | (b1 & 0xffff0000u);
        v[j] = (both & m) | (v[j] & ~m);
    }
}

__global__ void __launch_bounds__(256) k_ct_tile(CtArgs a)
{
    CtRow t;
    if (!ct_row(a, t)) return;
    ct_load(a, t);
    uint64_t edge, strong;
    ct_masks(t, edge, strong);
    const uint64_t reached = ct_grow(strong, edge);
    const uint64_t left = edge & ~reached;
    const uint64_t undecided = ct_grow((t.row == 0 || t.row == t.th - 1) ? left : left & (1ull | (1ull << ((t.tw - 1) & 63))), left);
    // settle the 127 pixels: reached -> 255, in no border-touching component -> 0, undecided stay
    ct_store(a, t, edge & ~strong & ~undecided, reached);

    // the mask of the tile's row 0 and of its last row, in all its lanes
    const auto top = [&](uint64_t m) { return ct_dpp64<0x150>(m); };
    const auto bottom = [&](uint64_t m) { return t.th == CT_H ? ct_dpp64<0x15f>(m) : __shfl(m, (t.lane & 48) + t.th - 1); };
    uint32_t topv[2] = {~0u, ~0u}, botv[2] = {~0u, ~0u}, leftv = CT_NONE, rightv = CT_NONE;
    const auto record = [&](uint64_t m, uint32_t code) {
        ct_codes(topv, top(m), t.row, code);
        ct_codes(botv, bottom(m), t.row, code);
        if (m & 1ull) leftv = code;
        if ((m >> ((t.tw - 1) & 63)) & 1ull) rightv = code;
    };
    record(reached, 0);
    gptr_t<uint32_t> par = gmem(a.parent);
    gptr_t<uint16_t> bt = gmem(a.border) + (long)t.tile * 2 * CT_NB;
    if (t.tile == 0 && t.row == 0) par[0] = 0;
    uint32_t k = 0;
    uint64_t bm = undecided;
    while (true) {
        const uint64_t live = __ballot(bm != 0ull);
        if (!live) break;
        const uint32_t mine = (uint32_t)(live >> (t.lane & 48)) & 0xffffu;   // the rows of my tile that hold some
        const bool first = (mine & (0u - mine)) == (1u << t.row);
        const uint64_t seed = first ? bm & (0ull - bm) : 0ull;
        const uint64_t c = ct_grow(seed, bm);
        if (first) {
            const uint32_t gid = 1u + (uint32_t)t.tile * CT_NB + k;
            par[gid] = gid;
            bt[CT_NB + k] = (uint16_t)(t.row * CT_W + __builtin_ctzll(seed));
        }
        record(c, k + 1);
        bm &= ~c;
        k += mine != 0;
    }
    if (t.in) {
        *(gptr_t<u32x2_dword>)(bt + 4 * t.row) = u32x2_dword{topv[0], topv[1]};
        *(gptr_t<u32x2_dword>)(bt + CT_W + 4 * t.row) = u32x2_dword{botv[0], botv[1]};
        bt[2 * CT_W + t.row] = (uint16_t)leftv;
        bt[2 * CT_W + CT_H + t.row] = (uint16_t)rightv;
        if (t.row == 0) gmem(a.ucount)[t.tile] = k;
    }
}

// the union-find id of a border code of a tile, -1 for none
MVX_DEV int32_t ct_id(int tile, uint32_t code)
{
    return code == CT_NONE ? -1 : code == 0 ? 0 : tile * CT_NB + (int32_t)code;
}

// the unions across the tile's right and bottom edges and its two lower corners: one wave per tile, all table
// reads first, so that the wave waits for memory once
__global__ void __launch_bounds__(256) k_ct_border(CtArgs a)
{
    const int lane = (int)threadIdx.x & 63;
    const int tile = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int tilesX = (int)a.tilesX;
    if (tile >= tilesX * (int)a.tilesY) return;
    const int tX = tile % tilesX, tY = tile / tilesX;
    const int tw = min(CT_W, (int)a.w - tX * CT_W), th = min(CT_H, (int)a.h - tY * CT_H);
    gptr_t<const uint16_t> bt = gmem((const uint16_t *)a.border) + (long)tile * 2 * CT_NB;
    gptr_t<const uint16_t> nr = bt + 2 * CT_NB, nd = bt + (long)tilesX * 2 * CT_NB;
    gptr_t<uint32_t> par = gmem(a.parent);
    // a right neighbour: this tile is full width; a lower one: it is full height, and that one of the same width
    const bool right = tX + 1 < tilesX, down = tY + 1 < (int)a.tilesY;
    const uint32_t ra = right && lane < th ? bt[2 * CT_W + CT_H + lane] : CT_NONE, rb = right && lane < th ? nr[2 * CT_W + lane] : CT_NONE;
    const uint32_t da = down && lane < tw ? bt[CT_W + lane] : CT_NONE, db = down && lane < tw ? nd[lane] : CT_NONE;
    const uint32_t cr = down && right ? (nd + 2 * CT_NB)[0] : CT_NONE, cl = down && tX > 0 ? (nd - 2 * CT_NB)[CT_W - 1] : CT_NONE;
    const int32_t d = ct_id(tile, da);
    const int32_t dr = __builtin_amdgcn_readlane(d, tw - 1), dl = __builtin_amdgcn_readlane(d, 0);
    border_unions(par, ct_id(tile, ra), ct_id(tile + 1, rb), lane);
    border_unions(par, d, ct_id(tile + tilesX, db), lane);
    if (lane == 0) {
        const int32_t qr = ct_id(tile + tilesX + 1, cr), ql = ct_id(tile + tilesX - 1, cl);
        if (dr >= 0 && qr >= 0) gunion(par, (uint32_t)dr, (uint32_t)qr);
        if (dl >= 0 && ql >= 0) gunion(par, (uint32_t)dl, (uint32_t)ql);
    }
}

// the undecided pixels of each tile: those of components whose root is the strong node, grown from the
// components' seeds, become 255, the others 0
__global__ void __launch_bounds__(256) k_ct_resolve(CtArgs a)
{
    __shared__ uint32_t seedLds[4][64][2];
    CtRow t;
    if (!ct_row(a, t)) return;
    const uint32_t count = t.in ? gmem((const uint32_t *)a.ucount)[t.tile] : 0u;
    if (!__any(count != 0u)) return;
    if (count == 0u) t.inner = 0ull;
    ct_load(a, t);
    uint32_t (&seeds)[64][2] = seedLds[threadIdx.x >> 6];
    seeds[t.lane][0] = seeds[t.lane][1] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (uint32_t k = (uint32_t)t.row; k < count; k += CT_H) {
        const uint32_t p = gmem((const uint16_t *)a.border)[(long)t.tile * 2 * CT_NB + CT_NB + k];
        if (gfind_settled<__HIP_MEMORY_SCOPE_WAVEFRONT>(gmem(a.parent), 1u + (uint32_t)t.tile * CT_NB + k) == 0u)
            atomicOr(&seeds[(t.lane & 48) + (int)(p / CT_W)][(p % CT_W) >> 5], 1u << (p & 31u));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint64_t edge, strong;
    ct_masks(t, edge, strong);
    const uint64_t weak = edge & ~strong;
    const uint64_t seed = ((uint64_t)seeds[t.lane][1] << 32) | seeds[t.lane][0];
    ct_store(a, t, weak, ct_grow(seed & weak, weak));
}

struct CtLayout { size_t parent, border, ucount, total; uint32_t tilesX, tilesY, quadsX, tiles; };

inline CtLayout ct_layout(uint32_t w, uint32_t h)
{
    CtLayout L;
    L.tilesX = (w + CT_W - 1) / CT_W;
    L.tilesY = (h + CT_H - 1) / CT_H;
    L.quadsX = (L.tilesX + CT_QUAD - 1) / CT_QUAD;
    L.tiles = L.tilesX * L.tilesY;
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    L.parent = 0;
    L.border = al(((size_t)L.tiles * CT_NB + 1) * 4);
    L.ucount = L.border + al((size_t)L.tiles * 2 * CT_NB * 2);
    L.total = L.ucount + al((size_t)L.tiles * 4);
    return L;
}

}  // namespace mvx

using namespace mvx;

namespace {
template <int G, bool L2>
int canny_sobel_g(mvx_stream_t stream, uint32_t w, uint32_t h, uint16_t *dst, uint32_t dstStride, const uint8_t *src,
                  uint32_t srcStride)
{
    if (w == 0 || h == 0) return MVX_SUCCESS;
    if (!plane_ok_c(dst, w, dstStride, 2) || !plane_ok_c(src, w, srcStride, 1)) return MVX_ERROR_INVALID_PARAMETERS;
    if ((int)h < G) return MVX_SUCCESS;
    // (the 3x3 L1 form takes larger planes too)
    if ((G != 3 || L2) && ((uint64_t)h * dstStride > 0xffffffffull || (uint64_t)h * srcStride > 0xffffffffull)) return MVX_ERROR_INVALID_PARAMETERS;
    if (w < 16) {
        hipLaunchKernelGGL((k_canny_sobel_g_narrow<G, L2>), dim3(1), dim3(64), 0, stream_of(stream), w, h, dst, dstStride, src, srcStride);
    } else {
        const uint32_t rows = h - 2 * (G / 2), units = ((w & ~15u) - 16) / 8, rowGroups = (rows + CSC_ROWS - 1) / CSC_ROWS;
        const uint32_t inner = (uint32_t)(((uint64_t)units * rowGroups + 255) / 256), edge = ((rows + CSW_ROWS - 1) / CSW_ROWS + 1) / 2;
        hipLaunchKernelGGL((k_canny_sobel_g<G, L2>), dim3(inner + edge), dim3(256), 0, stream_of(stream), w, h, dst, dstStride, src,
                           srcStride, edge, units, rowGroups);
    }
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}
}  // namespace

#define MVX_CANNY_SOBEL(NAME, G, L2)                                                                                      \
    extern "C" int NAME(mvx_stream_t stream, uint32_t w, uint32_t h, uint16_t *dst, uint32_t dstStride, const uint8_t *src, \
                        uint32_t srcStride)                                                                               \
    {                                                                                                                     \
        return canny_sobel_g<G, L2>(stream, w, h, dst, dstStride, src, srcStride);                                         \
    }
MVX_CANNY_SOBEL(mvx_CannySobel_U16_U8_3x3_L1NORM, 3, false)
MVX_CANNY_SOBEL(mvx_CannySobel_U16_U8_5x5_L1NORM, 5, false)
MVX_CANNY_SOBEL(mvx_CannySobel_U16_U8_7x7_L1NORM, 7, false)
MVX_CANNY_SOBEL(mvx_CannySobel_U16_U8_3x3_L2NORM, 3, true)
MVX_CANNY_SOBEL(mvx_CannySobel_U16_U8_5x5_L2NORM, 5, true)
MVX_CANNY_SOBEL(mvx_CannySobel_U16_U8_7x7_L2NORM, 7, true)
#undef MVX_CANNY_SOBEL

extern "C" int mvx_CannySuppThreshold_U8XY_U16_3x3(mvx_stream_t stream, uint32_t w, uint32_t h, uint8_t *dst,
                                                   uint32_t dstStride, const uint16_t *mag, uint32_t magStride,
                                                   void *xyStack, uint32_t capacityOfXY, uint32_t lower, uint32_t upper)
{
    if (w == 0 || h == 0) return MVX_SUCCESS;
    if (!plane_ok_c(dst, w, dstStride, 1) || !plane_ok_c(mag, w, magStride, 2) || !xyStack ||
        (uint64_t)capacityOfXY < (uint64_t)w * h)
        return MVX_ERROR_INVALID_PARAMETERS;
    if (w < 3 || h < 3) return MVX_SUCCESS;
    // a lower threshold above the upper one decides nothing: what is not above the upper is not above it either
    const auto plus1 = [](int32_t t) { return (uint32_t)(std::min(std::max(t, -1), 16383) + 1); };
    const int32_t lowerT = std::min((int32_t)lower, (int32_t)upper);
    const uint32_t units = (w + 7) / 8, rowGroups = (h - 2 + SUP_ROWS - 1) / SUP_ROWS;
    hipLaunchKernelGGL(k_canny_supp, dim3((uint32_t)(((uint64_t)units * rowGroups + 255) / 256)), dim3(256), 0, stream_of(stream), w, h,
                       dst, dstStride, mag, magStride, plus1(lowerT), plus1((int32_t)upper), units, rowGroups);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}

extern "C" int mvx_CannyEdgeTrace_U8_U8XY(mvx_stream_t stream, uint32_t w, uint32_t h, uint8_t *img, uint32_t stride,
                                          void *xyStack, uint32_t capacityOfXY)
{
    if (w == 0 || h == 0) return MVX_SUCCESS;
    // the stack holds 4-byte items (two 16-bit coordinates); both traces keep 32-bit words in it
    if (!plane_ok_c(img, w, stride, 1) || !xyStack || ((uintptr_t)xyStack & 3u) || (uint64_t)capacityOfXY < (uint64_t)w * h)
        return MVX_ERROR_INVALID_PARAMETERS;
    if (w < 3 || h < 3) return MVX_SUCCESS;
    const CtLayout L = ct_layout(w, h);
    if (L.total <= (size_t)capacityOfXY * 4) {
        // the tiled trace, its tables in the stack's memory (about 1.25 bytes per pixel)
        uint8_t *ws = (uint8_t *)xyStack;
        CtArgs a{w, h, stride, L.tilesX, L.tilesY, L.quadsX, img, (uint32_t *)(ws + L.parent), (uint16_t *)(ws + L.border),
                 (uint32_t *)(ws + L.ucount)};
        const dim3 quads((L.quadsX * L.tilesY + 3) / 4), grid((L.tiles + 3) / 4);
        hipLaunchKernelGGL(k_ct_tile, quads, dim3(256), 0, stream_of(stream), a);
        hipLaunchKernelGGL(k_ct_border, grid, dim3(256), 0, stream_of(stream), a);
        hipLaunchKernelGGL(k_ct_resolve, quads, dim3(256), 0, stream_of(stream), a);
        MVX_LAUNCH_CHECK();
        return MVX_SUCCESS;
    }
    // small images: a union-find over every interior edge pixel, the labels in the stack (4 bytes per pixel)
    dim3 grid((w - 2 + 255) / 256, h - 2);
    uint32_t *lab = (uint32_t *)xyStack;
    hipLaunchKernelGGL(k_canny_init, grid, dim3(256), 0, stream_of(stream), w, h, img, stride, lab);
    hipLaunchKernelGGL(k_canny_merge, grid, dim3(256), 0, stream_of(stream), w, h, img, stride, lab);
    hipLaunchKernelGGL(k_canny_mark, grid, dim3(256), 0, stream_of(stream), w, h, img, stride, lab);
    hipLaunchKernelGGL(k_canny_final, grid, dim3(256), 0, stream_of(stream), w, h, img, stride, lab);
    MVX_LAUNCH_CHECK();
    return MVX_SUCCESS;
}
