// probe_arith.hip -- test-only probes (libprobe_arith.so, loaded by tests/test_gpu_arith_exhaustive.py):
// exhaustive device-side comparisons of the Magnitude / Phase building blocks of the product
// kernels (mivisionx_amd/csrc/arith.hpp) against the operations they stand in for, over their
// whole input domains.
//   * div_small_rn(a, b) vs IEEE single division (__fdiv_rn), all integers 0 <= a <= b <= 32768;
//   * mag_body(gx, gy) vs rint(sqrt((double)(gx^2 + gy^2))) saturated to 32767 -- the reference's
//     cvtpd_epi32(sqrt_pd(.)) and packs (ago_haf_cpu_arithmetic.cpp:5031-5078) -- for all
//     0 <= gy <= gx <= 32768 (the result depends on |gx|, |gy| only);
//   * div_by_const_rn(a, b, RN(1/b)) vs IEEE single division for every finite float a, for a given b;
//   * l2_pack_simd(f) vs the Canny L2 SSE rule, cvtps_epi32(sqrt_ps(f)) packed to 16 bits, for every
//     integer-valued float below 2^32;
//   * mag_sobel, mag_sobel_trunc and phase_sobel vs mag_body and mag_tail, mag_trunc and phase_px, for every
//     pair of 3x3 Sobel gradients (-1020..1020 each);
//   * recip_usual(z) vs IEEE single division 1 / z, every mantissa at three exponents, and div_by(n, z, .) vs n / z,
//     every mantissa of z with a few hundred million dividends;
//   * the lane mapping of the DPP wave_shl:1 control.
#include "../../mivisionx_amd/csrc/arith.hpp"

using namespace mvx;

__global__ void k_div(uint32_t maxB, uint32_t *out)
{
    const uint32_t b = blockIdx.x + 1;
    if (b > maxB) return;
    for (uint32_t a = threadIdx.x; a <= b; a += blockDim.x) {
        const float q = div_small_rn((float)a, (float)b);
        const float r = __fdiv_rn((float)a, (float)b);
        if (__float_as_uint(q) != __float_as_uint(r)) {
            atomicAdd(out, 1u);
            atomicCAS(out + 1, 0u, (b << 16) | a);
        }
    }
}

__global__ void k_mag(uint32_t maxA, uint32_t *out)
{
    const uint32_t gx = blockIdx.x;
    if (gx > maxA) return;
    for (uint32_t gy = threadIdx.x; gy <= gx; gy += blockDim.x) {
        const int32_t m = mag_body((int32_t)gx, (int32_t)gy);
        const double s = (double)gx * gx + (double)gy * gy;
        const int32_t want = (int32_t)min(rint(sqrt(s)), 32767.0);
        if (m != want) {
            atomicAdd(out, 1u);
            atomicCAS(out + 1, 0u, (gx << 16) | gy);
        }
    }
}

__global__ void k_sobel_px(uint32_t maxG, uint32_t *out)
{
    const int32_t gx = (int32_t)blockIdx.x - (int32_t)maxG;
    for (int32_t gy = (int32_t)threadIdx.x - (int32_t)maxG; gy <= (int32_t)maxG; gy += (int32_t)blockDim.x) {
        const float fx = (float)gx, fy = (float)gy;
        const int32_t m = (int32_t)(mag_sobel(fx, fy) & 0xffffu);
        if (m != mag_body(gx, gy) || m != mag_tail(gx, gy) || (int32_t)mag_sobel_trunc(fx, fy) != mag_trunc(gx, gy) ||
            (phase_sobel(fx, fy) & 0xffu) != phase_px(gx, gy)) {
            atomicAdd(out, 1u);
            atomicCAS(out + 1, 0u, ((uint32_t)(gx + (int32_t)maxG) << 16) | (uint32_t)(gy + (int32_t)maxG));
        }
    }
}

static int run(void (*kernel)(uint32_t, uint32_t *), uint32_t blocks, uint32_t arg, uint32_t *result)
{
    uint32_t *d = nullptr;
    if (hipMalloc(&d, 8) != hipSuccess) return -1;
    int rc = -1;
    if (hipMemset(d, 0, 8) == hipSuccess) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, 0, arg, d);
        if (hipGetLastError() == hipSuccess && hipMemcpy(result, d, 8, hipMemcpyDeviceToHost) == hipSuccess) rc = 0;
    }
    (void)hipFree(d);
    return rc;
}

// a / norm by div_by_const_rn against IEEE division for every finite float a (2^32 - 2^24 inputs)
__global__ void k_div_const(float b, float y, uint32_t *out)
{
    const uint64_t base = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 256u;
    for (uint32_t k = 0; k < 256; k++) {
        const uint32_t bits = (uint32_t)(base + k);
        if (((bits >> 23) & 0xffu) == 0xffu) continue;   // Inf and NaN
        const float a = __uint_as_float(bits);
        const float q = div_by_const_rn(a, b, y), r = __fdiv_rn(a, b);
        if (__float_as_uint(q) != __float_as_uint(r)) {
            atomicAdd(out, 1u);
            atomicCAS(out + 1, 0u, bits);
        }
    }
}

// every mantissa of z in [2^e, 2^(e+1)): the reciprocal, and 64 quotients each
__global__ void k_recip(uint32_t e, uint32_t *out)
{
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= 1u << 23) return;
    const float z = __uint_as_float((e << 23) | m), r = recip_usual(z);
    bool same = __float_as_uint(r) == __float_as_uint(__fdiv_rn(1.f, z));
    uint32_t s = m * 2654435761u + e;
    for (int k = 0; k < 64; k++) {
        s = s * 1664525u + 1013904223u;
        const float n = __uint_as_float((s & 0x807fffffu) | ((100u + ((s >> 23) & 0x3fu)) << 23));   // 2^-27 .. 2^36, both signs
        same = same && div_by(n, z, r) == __fdiv_rn(n, z);
    }
    if (!same) {
        atomicAdd(out, 1u);
        atomicCAS(out + 1, 0u, m);
    }
}

// l2_pack_simd(f) against _mm_cvtps_epi32(_mm_sqrt_ps(f)) + unsigned 16-bit pack restated in double
// (the float square root is the double one rounded to float: double rounding is innocuous for sqrt),
// for f = (float)i, every integer 0 <= i < 2^32 (every integer-valued float below 2^32)
__global__ void k_l2pack(uint32_t *out)
{
    const uint64_t base = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 256u;
    for (uint32_t k = 0; k < 256; k++) {
        const uint32_t i = (uint32_t)(base + k);
        const float f = (float)i;
        const float r = (float)sqrt((double)f);
        const double want = fmin(rint((double)r), 65535.0);
        if (l2_pack_simd(f) != (int)want) {
            atomicAdd(out, 1u);
            atomicCAS(out + 1, 0u, i);
        }
    }
}

// lane i of wave_shl:1 (DPP control 0x130) reads lane i + 1; lane 63 reads nothing (0)
__global__ void k_dpp(int32_t *out)
{
    const int v = (int)threadIdx.x + 1000;
    out[threadIdx.x] = __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true);
}

// result[0] = mismatches, result[1] = first mismatch packed as (b << 16) | a (b, a <= 32768)
extern "C" int probe_div_small(uint32_t maxB, uint32_t *result) { return run(k_div, maxB, maxB, result); }
extern "C" int probe_recip(uint32_t e, uint32_t *result) { return run(k_recip, 1u << 15, e, result); }
extern "C" int probe_sobel_px(uint32_t maxG, uint32_t *result) { return run(k_sobel_px, 2 * maxG + 1, maxG, result); }
extern "C" int probe_mag_body(uint32_t maxA, uint32_t *result) { return run(k_mag, maxA + 1, maxA, result); }

// result[0] = mismatches, result[1] = bits of the first mismatching dividend
extern "C" int probe_div_const(float b, uint32_t *result)
{
    uint32_t *d = nullptr;
    if (hipMalloc(&d, 8) != hipSuccess) return -1;
    int rc = -1;
    if (hipMemset(d, 0, 8) == hipSuccess) {
        hipLaunchKernelGGL(k_div_const, dim3(65536), dim3(256), 0, 0, b, recip_rn(b), d);   // 2^32 / 256 threads
        if (hipGetLastError() == hipSuccess && hipMemcpy(result, d, 8, hipMemcpyDeviceToHost) == hipSuccess) rc = 0;
    }
    (void)hipFree(d);
    return rc;
}

// result[0] = mismatches, result[1] = the first mismatching integer
extern "C" int probe_l2_pack(uint32_t *result)
{
    uint32_t *d = nullptr;
    if (hipMalloc(&d, 8) != hipSuccess) return -1;
    int rc = -1;
    if (hipMemset(d, 0, 8) == hipSuccess) {
        hipLaunchKernelGGL(k_l2pack, dim3(65536), dim3(256), 0, 0, d);   // 2^32 / 256 threads
        if (hipGetLastError() == hipSuccess && hipMemcpy(result, d, 8, hipMemcpyDeviceToHost) == hipSuccess) rc = 0;
    }
    (void)hipFree(d);
    return rc;
}

// out[64]: what each lane of one wave reads through wave_shl:1
extern "C" int probe_dpp_wave_shl1(int32_t *out)
{
    int32_t *d = nullptr;
    if (hipMalloc(&d, 64 * sizeof(int32_t)) != hipSuccess) return -1;
    int rc = -1;
    hipLaunchKernelGGL(k_dpp, dim3(1), dim3(64), 0, 0, d);
    if (hipGetLastError() == hipSuccess && hipMemcpy(out, d, 64 * sizeof(int32_t), hipMemcpyDeviceToHost) == hipSuccess) rc = 0;
    (void)hipFree(d);
    return rc;
}
