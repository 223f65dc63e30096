// split_common.h -- the exact three-part bf16 split and its MFMAs (gfx950),
// and the layout of k_screen's centre image, shared by split_kernels.hip and
// screen_kernels.hip.
#pragma once

#include "fused_common.h"

namespace skm {

// ---------------------------------------------------------------------------
// Three-part bf16 split.  bf16 keeps fp32's exponent range with 8 significant
// bits, so every finite fp32 v with |v| >= 2^-103 is the exact sum of three
// bf16 values, each rounded to nearest:
//   hi = bf16(v),  mid = bf16(v - hi),  lo = (v - hi) - mid.
// v - hi is a multiple of v's fp32 ulp no larger than 2^16 of them, so the fp32
// subtraction is exact; likewise (v - hi) - mid, which is at most 2^8 ulps and
// therefore exactly a bf16.  |mid| <= 2^-8 |v|, |lo| <= 2^-16 |v|.
// A product of two bf16 values is exact in fp32, and the MFMAs accumulate in
// fp32, so
//  - the per-cluster sums (one-hot x hi, x mid, x lo) add every x exactly as
//    given, in fp32 (the one-hot operand is exact);
//  - the E-step takes 6 of the 9 part products of x.c (hh, hm, mh, hl, lh, mm):
//    the three left out (ml, lm, ll) total at most (2^-23 + 2^-32) |x_i c_i|
//    per feature, two units of fp32 roundoff, against the one unit by which an
//    fp32 product of x_i and c_i is itself rounded.

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

// (a, b) rounded to nearest even bf16, a in the low half: v_cvt_pk_bf16_f32
__device__ __forceinline__ unsigned pack_bf16(float a, float b)
{
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, v2bf));
}

__device__ __forceinline__ float bf16_lo(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

// The parts of a and b, as bf16 pairs (a's part in the low half).
__device__ __forceinline__ void split3(float a, float b, unsigned& hi, unsigned& mid, unsigned& lo)
{
    hi = pack_bf16(a, b);
    const float ra = a - bf16_lo(hi), rb = b - bf16_hi(hi);  // exact
    mid = pack_bf16(ra, rb);
    lo = pack_bf16(ra - bf16_lo(mid), rb - bf16_hi(mid));   // exact, and exactly bf16
}

struct Parts8 {
    v8bf h, m, l;
};
struct Parts4 {
    v4s h, m, l;  // 16x16x16 bf16 operands are passed as shorts
};

__device__ __forceinline__ Parts8 split8(float4 u, float4 v)
{
    unsigned h0, h1, h2, h3, m0, m1, m2, m3, l0, l1, l2, l3;
    split3(u.x, u.y, h0, m0, l0);
    split3(u.z, u.w, h1, m1, l1);
    split3(v.x, v.y, h2, m2, l2);
    split3(v.z, v.w, h3, m3, l3);
    return Parts8{__builtin_bit_cast(v8bf, v4u{h0, h1, h2, h3}), __builtin_bit_cast(v8bf, v4u{m0, m1, m2, m3}),
                  __builtin_bit_cast(v8bf, v4u{l0, l1, l2, l3})};
}

__device__ __forceinline__ Parts4 split4(float4 u)
{
    unsigned h0, h1, m0, m1, l0, l1;
    split3(u.x, u.y, h0, m0, l0);
    split3(u.z, u.w, h1, m1, l1);
    return Parts4{__builtin_bit_cast(v4s, v2u{h0, h1}), __builtin_bit_cast(v4s, v2u{m0, m1}),
                  __builtin_bit_cast(v4s, v2u{l0, l1})};
}

// D += A B on bf16: 16x16x32 (8 values per lane) and 16x16x16 (4)
__device__ __forceinline__ v4f mfma_bf16(v8bf a, v8bf b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma_bf16(v4s a, v4s b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// acc += the six kept part products of a.b (smaller terms first)
template <typename P>
__device__ __forceinline__ v4f dot6(const P& a, const P& b, v4f acc)
{
    acc = mfma_bf16(a.m, b.m, acc);
    acc = mfma_bf16(a.l, b.h, acc);
    acc = mfma_bf16(a.h, b.l, acc);
    acc = mfma_bf16(a.m, b.h, acc);
    acc = mfma_bf16(a.h, b.m, acc);
    return mfma_bf16(a.h, b.h, acc);
}

// Rows of 32 NK bf16 (the high parts; NK K32 steps) of kScreenSC centres a
// stage, padded to an odd number of 16-byte units, then -||c||^2 / 2 of the
// stage's centres (-3e38 for padding centres: they never lead) and the
// largest ||c||^2 of the stage as float bits (NaN counts above every number).
template <int NK>
struct ScreenGeom {
    static constexpr int CSTR = 32 * NK + 8;
    static constexpr int PBYTES = kScreenSC * CSTR * 2;
    static constexpr int STAGE = (PBYTES + kScreenSC * 4 + 16 + 1023) / 1024 * 1024;
    static constexpr int RES = (160 * 1024 - 256) / STAGE;  // stages that LDS holds
};

// Stage b of k_screen's image, by a block of 256 threads.
template <int NK>
__device__ __forceinline__ void screen_image(const float* __restrict__ C, const float* __restrict__ cnorm, int k,
                                             int ld, char* __restrict__ img, int b)
{
    using G = ScreenGeom<NK>;
    __shared__ unsigned sMax;
    const int tid = threadIdx.x, j0 = b * kScreenSC;
    char* const out = img + (size_t)b * G::STAGE;
    if (tid == 0) sMax = 0u;
    __syncthreads();
    constexpr int Q = G::CSTR / 4;
    for (int e = tid; e < kScreenSC * Q; e += 256) {
        const int c = e / Q, f = 4 * (e - c * Q);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (f < ld && j0 + c < k) v = *reinterpret_cast<const float4*>(C + (long)(j0 + c) * ld + f);
        *reinterpret_cast<v2u*>(out + (c * G::CSTR + f) * 2) = v2u{pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
    }
    float* const sn = reinterpret_cast<float*>(out + G::PBYTES);
    if (tid < kScreenSC) {
        const int j = j0 + tid;
        const float cn = j < k ? cnorm[j] : 0.f;
        sn[tid] = j < k ? -0.5f * cn : -3e38f;
        atomicMax(&sMax, __float_as_uint(cn) & 0x7fffffffu);
    }
    __syncthreads();
    if (tid == 0) reinterpret_cast<unsigned*>(sn)[kScreenSC] = sMax;
}

// Stage b = cg nks + ks of k_screen_wide's image, by a block of 256 threads:
// features 64 ks.. of centres 256 cg.. as rows of 64 bf16 (the high parts),
// padded to 72; after the last stage, -||c||^2 / 2 of every centre (-3e38
// past k).
constexpr int kWideStr = 72;                       // bf16 per LDS row: an odd number of 16-byte units
constexpr int kWideStage = 256 * kWideStr * 2;     // bytes
__device__ __forceinline__ void wide_image(const float* __restrict__ C, const float* __restrict__ cnorm, int k, int ld,
                                           char* __restrict__ img, int b)
{
    const int nks = (ld + 63) / 64, cg = b / nks, ks = b - cg * nks, ncg = (k + 255) / 256;
    __bf16* const out = reinterpret_cast<__bf16*>(img + (size_t)b * kWideStage);
    for (int e = threadIdx.x; e < 256 * 16; e += 256) {
        const int c = e >> 4, q = e & 15, j = 256 * cg + c, f = 64 * ks + 4 * q;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < k && f < ld) v = *reinterpret_cast<const float4*>(C + (long)j * ld + f);
        *reinterpret_cast<v2u*>(out + c * kWideStr + 4 * q) = v2u{pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
    }
    if (ks == 0) {
        const int j = 256 * cg + threadIdx.x;
        float* const ini = reinterpret_cast<float*>(img + (size_t)ncg * nks * kWideStage);
        ini[j] = j < k ? -0.5f * cnorm[j] : -3e38f;
    }
}

}  // namespace skm
