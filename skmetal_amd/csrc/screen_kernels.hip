// screen_kernels.hip -- a certified screen in front of the split E-step
// (gfx950).
//
// k_assign3 takes six bf16 part products for every x.c and is bound by them.
// For most rows one of the six settles the label: the product of the high
// parts, hh, differs from the six-product value by less than
//   e = 1.05 (2^-7 + ..) ||x|| max ||c||   (screen_slack below),
// so when a row's largest hh.. value leads its second largest by more than
// 2 e, the six products have their first minimum at the same centre, and no
// other centre can tie with it.  k_screen labels those rows and leaves the
// others' bits in `masks`; k_assign3_list (split_kernels.hip) then runs the
// six products for these rows alone.  Labels are those of k_assign3, bit for
// bit, whatever the data.
#include "split_common.h"

namespace skm {

// A bound on how far a screen value lies from x.c - ||c||^2 / 2 as the six
// products give it, for a row with ||x||^2 = xx (fp32 sum) and C2 = the
// largest ||c||^2, ldp features with the padding:
//   rounding x and c to bf16, 2^-8 of each value at most (8 significant bits),
//   and the index in the low six or seven bits: 2^-7 + 2^-16 + 2^-16 of
//   ||x|| ||c||; the screen's fp32 accumulation, ldp + 1
//   terms, and the six products', 6 ldp terms, at most 2^-23 of the terms'
//   magnitudes each (the terms of one row and centre total at most ||x||
//   ||c|| by Cauchy-Schwarz); the products left out, 2^-22; the same for
//   ||c||^2 / 2; and what a flush of subnormal parts and products can take.
// The factor 1.05 covers the norms' own rounding, and ldp 2^-125 what their
// squares lose below the smallest normal number (centres of 2^-80 have
// ||c||^2 = 0 in fp32, but products with rows of order 1 that the six products
// tell apart).
__device__ __forceinline__ float screen_slack(float xx, float C2, int ldp)
{
    const float lost = (float)ldp * 0x1p-125f;
    const float xn = sqrtf(xx + lost), cn = sqrtf(C2 + lost);
    const float a = 0x1p-7f + 0x1p-14f + 8.f * (float)ldp * 0x1p-23f;
    const float b = 0x1p-15f + (float)(ldp + 2) * 0x1p-23f;
    return 1.05f * (a * xn * cn + b * 0.5f * C2) + 0x1p-100f * (xn + cn) + 0x1p-100f;
}

// The largest of three: fmaxf would quiet each operand with an instruction of
// its own first.  (Its operands are VALU results, never an MFMA's.)
__device__ __forceinline__ float max3(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// D += A B on bf16, 32x32x16: lane l holds A[m = l%32][kk = 8(l/32) + j] and
// B[kk = 8(l/32) + j][n = l%32], j < 8, and receives D[m = 8(i/4) + 4(l/32) +
// i%4][n = l%32], i < 16.
typedef float v16f __attribute__((ext_vector_type(16)));
__device__ __forceinline__ v16f mfma32_bf16(v8bf a, v8bf b, v16f c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// A lane's 16 values of a block into its two largest, places p0.. of the
// stage in their low six bits.
__device__ __forceinline__ void two_largest(float& m1, float& m2, const v16f& acc, int p0)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            u[i] = __uint_as_float((__float_as_uint(acc[4 * q + i]) & ~63u) | (unsigned)(p0 + 4 * q + i));
        // with m1 >= m2 the second largest of m1, m2 and two more is the
        // larger of m2 and the middle one of the rest
        const float a1 = __builtin_amdgcn_fmed3f(m1, u[0], u[1]);
        m1 = max3(m1, u[0], u[1]);
        const float a2 = __builtin_amdgcn_fmed3f(m1, u[2], u[3]);
        m1 = max3(m1, u[2], u[3]);
        m2 = max3(m2, a1, a2);
    }
    // the values are used up here: sunk to the end of the stage they spill
    asm volatile("" : "+v"(m1), "+v"(m2));
}

// The centre of place p of a 128-centre stage, for a lane with h = lane / 32.
__device__ __forceinline__ int place_centre(int p, int h)
{
    return 32 * (p >> 4) + 8 * ((p & 15) >> 2) + 4 * h + (p & 3);
}

// A wave takes 64 rows at a time, in two 32-row groups whose high parts stay
// in registers (rows of at most 128 floats) while the centres pass by in LDS
// stages of kScreenSC: all of them resident, and the waves free to drift
// apart, where LDS holds them, else the next stage copied in with
// direct-to-LDS loads while the current one is used.  Each 32 x 32 tile's
// MFMAs are issued before the values of the tile before it are taken.  Per 32 centres a wave
// reads 2 NK 1 KB operands for 4 NK MFMAs; the accumulators start from
// -||c||^2 / 2, so that they end as the value to maximise.  Lane l keeps the
// two largest over its centres of row l%32 of each group, the centre's place
// in the stage in the low six bits of the value: nine VALU instructions for
// four values.  MFMAs and VALU instructions hardly overlap here, whether of
// one wave or of several: 8 16x16x32 MFMAs and 36 v_max3 take 57 and 65 ns a
// wave and SIMD alone, 106 together; the same work in 32x32x16 MFMAs 81.
// So the rows' K steps take features 32 s + 16 (l/32) + 8 t + j: each lane's
// 64 bytes of a row in a row.
// As many waves as the registers leave (2M x 64, k = 1,024: 281 us with
// twelve, 290 with eight and both groups of the next rows in flight; 1M x 128,
// k = 256: sixteen without prefetch 149, eight with 107).
constexpr int screen_waves(int nk) { return nk <= 2 ? 12 : 8; }
template <int NK>
__global__ __launch_bounds__(64 * screen_waves(NK), screen_waves(NK) / 4) void k_screen(ScreenArgs a, int resident)
{
    using G = ScreenGeom<NK>;
    constexpr int NW = screen_waves(NK);
    if (a.state != nullptr && a.state->done != 0) return;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ int sChg;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r32 = lane & 31;
    const int ld = a.ld;
    const long n = a.n;
    if (tid == 0) sChg = 0;
    int nchg = 0;
    const int nst = (a.k + kScreenSC - 1) / kScreenSC;
    const int stage_bytes = G::STAGE;
    const __amdgpu_buffer_rsrc_t irs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.img), (short)0, nst * stage_bytes, 0x00020000);
    auto copy_stage = [&](int stg, int b) {
        char* dst = smem + b * stage_bytes;
        for (int i = wave; i < stage_bytes / 1024; i += NW) {
            const int soff = stg * stage_bytes + i * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(irs, (__attribute__((address_space(3))) void*)(dst + i * 1024), 16,
                                                     lane * 16, soff, 0, 0);
        }
    };
    if (resident)
        for (int stg = 0; stg < nst; ++stg) copy_stage(stg, stg);
    else
        copy_stage(0, 0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int cur = 0;
    // (resident: a wave stops at its own last rows; else all waves take part
    // in the stages of the block's)
    const long wstep = (long)gridDim.x * (64 * NW);
    auto rows_at = [&](long base) { return resident ? base : base + (long)gridDim.x * 64 * wave; };
    auto rows_rsrc = [&](long wrow) {
        const long nrow = n - wrow < 64 ? (n - wrow > 0 ? n - wrow : 0) : 64;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.X + (nrow > 0 ? wrow * ld : 0)), (short)0,
                                                 (int)(nrow * ld * 4), 0x00020000);
    };
    // group g's rows (a lane past the rows' end loads 0, one past a row's end
    // the next row's values: these meet zero centre parts and are kept out of
    // the norm).  Group 0 of the next 64 rows is in flight while the current
    // ones meet the centres: registers for no more.
    f4v raw[NK][4];
    auto load = [&](f4v(&q)[NK][4], __amdgpu_buffer_rsrc_t rs, int g) {
#pragma unroll
        for (int s = 0; s < NK; ++s) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(
                    rs, ((32 * g + r32) * ld + 32 * s + 16 * h + 4 * t) * 4, 0, 0);
                q[s][t] = __builtin_bit_cast(f4v, v);
            }
        }
    };
    const long first = (long)blockIdx.x * 64 + (resident ? (long)gridDim.x * 64 * wave : 0);
    load(raw, rows_rsrc(rows_at(first)), 0);
    for (long base = first; base < n; base += wstep) {
        const long wrow = rows_at(base);
        const long nrow = n - wrow < 64 ? (n - wrow > 0 ? n - wrow : 0) : 64;
        // the rows' high parts and ||x||^2
        v8bf xh[2][2 * NK];
        float xx[2];
        auto parts = [&](const f4v(&q)[NK][4], int g) {
            xx[g] = 0.f;
#pragma unroll
            for (int s = 0; s < NK; ++s) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float in = 32 * s + 16 * h + 4 * t < ld ? 1.f : 0.f;
                    const f4v v = q[s][t];
                    xx[g] = fmaf(fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))), in, xx[g]);
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f4v u = q[s][2 * t], v = q[s][2 * t + 1];
                    xh[g][2 * s + t] = __builtin_bit_cast(v8bf, v4u{pack_bf16(u.x, u.y), pack_bf16(u.z, u.w),
                                                                    pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)});
                }
            }
            // the norm is taken here (sunk to its use it keeps the fp32 row
            // alive)
            asm volatile("" : "+v"(xx[g]));
        };
        parts(raw, 0);
        load(raw, rows_rsrc(wrow), 1);
        parts(raw, 1);
        if (base + wstep < n) load(raw, rows_rsrc(rows_at(base + wstep)), 0);
        __builtin_amdgcn_sched_barrier(0);
        float m1[2], m2[2];
        int ms[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            m1[g] = m2[g] = -INFINITY;
            ms[g] = 0;
        }
        unsigned cmax = 0u;
        auto take = [&](int g, const v16f& acc, int cb) { two_largest(m1[g], m2[g], acc, 16 * cb); };
        v16f late;  // group 1 of the block before
#pragma unroll
        for (int i = 0; i < 16; ++i) late[i] = -3e38f;
        float was[2] = {m1[0], m1[1]};
        for (int stg = 0; stg < nst; ++stg) {
            if (!resident) copy_stage(stg + 1 < nst ? stg + 1 : 0, cur ^ 1);
            const char* const sb = smem + (resident ? stg : cur) * stage_bytes;
            const __bf16* const cb0 = reinterpret_cast<const __bf16*>(sb) + r32 * G::CSTR + 16 * h;
            const float* const sn = reinterpret_cast<const float*>(sb + G::PBYTES);
            cmax = max(cmax, reinterpret_cast<const unsigned*>(sn)[kScreenSC]);
            constexpr int NB = kScreenSC / 32;
#pragma unroll
            for (int cb = 0; cb < NB; ++cb) {
                v16f init;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4f c4 = *reinterpret_cast<const v4f*>(sn + 32 * cb + 8 * q + 4 * h);
#pragma unroll
                    for (int i = 0; i < 4; ++i) init[4 * q + i] = c4[i];
                }
                auto centres = [&](int s) {
                    return *reinterpret_cast<const v8bf*>(cb0 + 32 * cb * G::CSTR + 32 * (s >> 1) + 8 * (s & 1));
                };
                v8bf ca[2 * NK];
#pragma unroll
                for (int s = 0; s < 2 * NK; ++s) ca[s] = centres(s);
                v16f acc = init;
#pragma unroll
                for (int s = 0; s < 2 * NK; ++s) acc = mfma32_bf16(ca[s], xh[0][s], acc);
                take(1, late, cb == 0 ? NB - 1 : cb - 1);
                if (cb == 0) {  // the stage before is through
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        ms[g] = m1[g] != was[g] ? stg - 1 : ms[g];
                        was[g] = m1[g];
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                late = init;
#pragma unroll
                for (int s = 0; s < 2 * NK; ++s) late = mfma32_bf16(ca[s], xh[1][s], late);
                take(0, acc, cb);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!resident) {
                // the next stage is in (every wave's copies) and this one is
                // read: swap
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
                cur ^= 1;
            }
        }
        take(1, late, kScreenSC / 32 - 1);
#pragma unroll
        for (int g = 0; g < 2; ++g) ms[g] = m1[g] != was[g] ? nst - 1 : ms[g];
        // the two lanes of a row; lane l keeps row l of the wave's 64
        float b1 = 0.f, b2 = 0.f, bx = 0.f;
        int bi = 0;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            int i1 = ms[g] * kScreenSC + place_centre((int)(__float_as_uint(m1[g]) & 63u), h);
            const float o1 = __shfl_xor(m1[g], 32), o2 = __shfl_xor(m2[g], 32);
            const int oi = __shfl_xor(i1, 32);
            const float x2 = xx[g] + __shfl_xor(xx[g], 32);
            const float d2 = fmaxf(fminf(m1[g], o1), fmaxf(m2[g], o2));
            i1 = o1 > m1[g] ? oi : i1;
            if (h == g) {
                b1 = fmaxf(m1[g], o1);
                b2 = d2;
                bi = i1;
                bx = x2;
            }
        }
        const float C2 = __uint_as_float(cmax);
        const float slack = screen_slack(bx, C2, 32 * NK);
        // (the magnitudes' bound keeps every sum finite; a NaN in the norms
        // fails it)
        const bool sure = (b1 - b2 > 2.f * slack) & (sqrtf(bx) * sqrtf(C2) + C2 < 1e37f);
        const bool valid = lane < nrow;
        const long row = wrow + lane;
        int moved = 0;
        if (valid && sure) {
            if (a.changed != nullptr) moved = a.labels[row] != bi;
            a.labels[row] = bi;
            if (a.emin != nullptr) a.emin[row] = -2.f * b1;
        }
        if (a.changed != nullptr) nchg += (int)__popcll(__ballot(moved));
        const unsigned long long left = __ballot(valid && !sure);
        if (lane == 0 && nrow > 0) a.masks[wrow >> 6] = left;
    }
    if (a.changed != nullptr) {
        if (lane == 0 && nchg != 0) atomicAdd(&sChg, nchg);
        __syncthreads();
        if (tid == 0 && sChg != 0) atomicAdd(a.changed, sChg);
    }
}

template <int NK>
static hipError_t launch_screen_nk(const ScreenArgs& a, int num_cu, hipStream_t s)
{
    using G = ScreenGeom<NK>;
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_screen<NK>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, G::RES * G::STAGE);
    if (e != hipSuccess) return e;
    const int nst = (a.k + kScreenSC - 1) / kScreenSC;
    const int resident = nst <= G::RES;
    constexpr int NW = screen_waves(NK);
    const long blocks = (a.n + 64 * NW - 1) / (64 * NW);
    hipLaunchKernelGGL(k_screen<NK>, dim3((unsigned)(blocks < num_cu ? blocks : num_cu)), dim3(64 * NW),
                       (size_t)(resident ? nst : 2) * G::STAGE, s, a, resident);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// rows of more than 128 floats
// ---------------------------------------------------------------------------
//
// A block: 256 rows x 256 centres, wave w the 64 rows 64 (w % 4).. against the
// 128 centres 128 (w / 4)..: eight 32 x 32 accumulators, six 1 KB operands for
// eight MFMAs a K16 step (LDS at 96 of its 128 bytes a cycle).  K goes by in
// stages of 64 features, two in LDS: while one is used, the next one's
// centres come in with direct-to-LDS loads, and its rows as fp32 into
// registers, rounded to bf16 on the way to LDS.  Blocks of one row block
// follow each other on one XCD (block b runs on XCD b % 8), so that X and the
// image come from its L2.  A launch takes wide_rows rows.
__global__ __launch_bounds__(512, 2) void k_screen_wide(WideArgs a)
{
    if (a.state != nullptr && a.state->done != 0) return;
    const int ncg = (a.k + 255) / 256, nks = (a.ld + 63) / 64;
    const long nrb = (a.n + 255) / 256;
    const long i = blockIdx.x >> 3;
    const long rb = (blockIdx.x & 7) + 8 * (i / ncg);
    const int cg = (int)(i % ncg);
    if (rb >= nrb) return;
    extern __shared__ __attribute__((aligned(1024))) char smem[];  // [2] rows, [2] centres
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r32 = lane & 31;
    const int ld = a.ld;
    const long r0 = rb * 256;
    const int nrow = (int)(a.n - r0 < 256 ? a.n - r0 : 256);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.X + r0 * ld), (short)0,
                                                                        nrow * ld * 4, 0x00020000);
    const int stage_bytes = kWideStage;
    const __amdgpu_buffer_rsrc_t irs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(a.img + (size_t)cg * nks * stage_bytes), (short)0, nks * stage_bytes, 0x00020000);
    auto copy_centres = [&](int ks, int b) {
        char* dst = smem + (2 + b) * stage_bytes;
        for (int q = wave; q < stage_bytes / 1024; q += 8) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(irs, (__attribute__((address_space(3))) void*)(dst + q * 1024), 16,
                                                     lane * 16, ks * stage_bytes + q * 1024, 0, 0);
        }
    };
    // the stage's rows: lane l of wave w loads float4 l % 16 of rows 32 w + 4 u
    // + l / 16 (past the rows' end 0, past a row's end the next row's values,
    // which meet zero centre parts)
    const int q16 = lane & 15, lr = 32 * wave + (lane >> 4);
    f4v raw[8];
    float xx[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) xx[u] = 0.f;
    auto load_rows = [&](int ks) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            raw[u] = __builtin_bit_cast(
                f4v, __builtin_amdgcn_raw_buffer_load_b128(rs, ((lr + 4 * u) * ld + 64 * ks + 4 * q16) * 4, 0, 0));
    };
    auto put_rows = [&](int ks, int b) {
        __bf16* dst = reinterpret_cast<__bf16*>(smem + b * stage_bytes);
        const float in = 64 * ks + 4 * q16 < ld ? 1.f : 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const f4v v = raw[u];
            *reinterpret_cast<v2u*>(dst + (lr + 4 * u) * kWideStr + 4 * q16) =
                v2u{pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
        }
        if (cg == 0) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const f4v v = raw[u];
                xx[u] = fmaf(fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))), in, xx[u]);
            }
        }
    };
    load_rows(0);
    copy_centres(0, 0);
    const int wr = wave & 3, wc = wave >> 2;
    // the accumulators start from -||c||^2 / 2
    const float* const ini =
        reinterpret_cast<const float*>(a.img + (size_t)ncg * nks * stage_bytes) + 256 * cg + 128 * wc + 4 * h;
    v16f acc[4][2];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f4v v = *reinterpret_cast<const f4v*>(ini + 32 * c + 8 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[c][0][4 * q + e] = v[e];
        }
        acc[c][1] = acc[c][0];
    }
    put_rows(0, 0);
    if (nks > 1) load_rows(1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int ks = 0; ks < nks; ++ks) {
        const int cur = ks & 1;
        if (ks + 1 < nks) {
            // the next stage: its rows, loaded a stage ago, to LDS, and its
            // centres; then the rows of the one after it (their wait at the
            // end of the stage left half of it idle)
            put_rows(ks + 1, cur ^ 1);
            copy_centres(ks + 1, cur ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            if (ks + 2 < nks) load_rows(ks + 2);
            __builtin_amdgcn_sched_barrier(0);
        }
        const __bf16* const xb =
            reinterpret_cast<const __bf16*>(smem + cur * stage_bytes) + (64 * wr + r32) * kWideStr + 8 * h;
        const __bf16* const cb =
            reinterpret_cast<const __bf16*>(smem + (2 + cur) * stage_bytes) + (128 * wc + r32) * kWideStr + 8 * h;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            v8bf x[2], c[4];
#pragma unroll
            for (int g = 0; g < 2; ++g) x[g] = *reinterpret_cast<const v8bf*>(xb + 32 * g * kWideStr + 16 * s);
#pragma unroll
            for (int e = 0; e < 4; ++e) c[e] = *reinterpret_cast<const v8bf*>(cb + 32 * e * kWideStr + 16 * s);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int g = 0; g < 2; ++g) acc[e][g] = mfma32_bf16(c[e], x[g], acc[e][g]);
            }
        }
        if (ks + 1 < nks) {
            // the next stage is in and this one is read: swap.  vmcnt(8):
            // everything but the eight row loads issued last (loads complete
            // in order); lgkmcnt(0): this wave's LDS writes.
            if (ks + 2 < nks)
                __builtin_amdgcn_s_waitcnt(0x0078);
            else
                __builtin_amdgcn_s_waitcnt(0);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_barrier();
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
        }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        float m1 = -INFINITY, m2 = -INFINITY;
#pragma unroll
        for (int c = 0; c < 4; ++c) two_largest(m1, m2, acc[c][g], 16 * c);
        // the two lanes of a row: the larger value carries the centre's place
        // among the 128 in its low seven bits
        const int id = place_centre((int)(__float_as_uint(m1) & 63u), h);
        m1 = __uint_as_float((__float_as_uint(m1) & ~127u) | (unsigned)id);
        const float o1 = __shfl_xor(m1, 32), o2 = __shfl_xor(m2, 32);
        m2 = fmaxf(fminf(m1, o1), fmaxf(m2, o2));
        m1 = fmaxf(m1, o1);
        const int r = 64 * wr + 32 * g + r32;
        if (h == 0 && r < nrow)
            reinterpret_cast<float2*>(a.part)[(long)(2 * cg + wc) * a.n + r0 + r] = make_float2(m1, m2);
    }
    if (cg == 0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            float t = xx[u];
            t += __shfl_xor(t, 1);
            t += __shfl_xor(t, 2);
            t += __shfl_xor(t, 4);
            t += __shfl_xor(t, 8);
            const int r = lr + 4 * u;
            if (q16 == 0 && r < nrow) a.xx[r0 + r] = t;
        }
    }
}

// A thread per row: the two largest over the parts, then the row's label or
// its place on the list.
__global__ __launch_bounds__(256) void k_screen_merge(WideArgs a)
{
    if (a.state != nullptr && a.state->done != 0) return;
    constexpr unsigned long long kNone = 0xff800000ull << 32;  // +inf in order_bits's form, centre 0
    const long row = (long)blockIdx.x * 256 + threadIdx.x;
    __shared__ unsigned sMax;
    __shared__ int sChg, sLeft, sAt;
    const int tid = threadIdx.x;
    if (tid == 0) {
        sMax = 0u;
        sChg = 0;
        sLeft = 0;
    }
    __syncthreads();
    unsigned cm = 0u;  // the largest ||c||^2 as bits: NaN counts above every number
    for (int j = tid; j < a.k; j += 256) cm = max(cm, __float_as_uint(a.cnorm[j]) & 0x7fffffffu);
    atomicMax(&sMax, cm);
    const int np = 2 * ((a.k + 255) / 256);
    float m1 = -INFINITY, m2 = -INFINITY;
    int mp = 0;
    const bool valid = row < a.n;
    if (valid) {
        for (int p = 0; p < np; ++p) {
            const float2 v = reinterpret_cast<const float2*>(a.part)[(long)p * a.n + row];
            m2 = fmaxf(fminf(m1, v.x), fmaxf(m2, v.y));
            if (v.x > m1) {
                m1 = v.x;
                mp = p;
            }
        }
    }
    __syncthreads();
    const float C2 = __uint_as_float(sMax), xx = valid ? a.xx[row] : 0.f;
    const float slack = screen_slack(xx, C2, 64 * ((a.ld + 63) / 64));
    const bool sure = (m1 - m2 > 2.f * slack) & (sqrtf(xx) * sqrtf(C2) + C2 < 1e37f);
    int at = 0;
    if (valid && sure) {
        const int lab = 128 * mp + (int)(__float_as_uint(m1) & 127u);
        if (a.changed != nullptr && a.labels[row] != lab) atomicAdd(&sChg, 1);
        a.labels[row] = lab;
    } else if (valid) {
        at = atomicAdd(&sLeft, 1);
        a.keys[row] = kNone;
    }
    __syncthreads();
    if (tid == 0) {
        if (a.changed != nullptr && sChg != 0) atomicAdd(a.changed, sChg);
        sAt = sLeft != 0 ? atomicAdd(a.nlist, sLeft) : 0;
    }
    __syncthreads();
    if (valid && !sure) a.list[sAt + at] = (unsigned)(a.row0 + row);
}

size_t wide_image_bytes(int k, int ld)
{
    const size_t ncg = size_t(k + 255) / 256, nks = size_t(ld + 63) / 64;
    return ncg * nks * kWideStage + ncg * 256 * sizeof(float);
}

hipError_t launch_screen_wide(const WideArgs& a, hipStream_t s)
{
    if (a.n <= 0) return hipSuccess;
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_screen_wide),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, 4 * kWideStage);
    if (e != hipSuccess) return e;
    const long rows = wide_rows(a.n, a.k);
    for (long r = 0; r < a.n; r += rows) {
        WideArgs b = a;
        b.row0 = r;
        b.n = a.n - r < rows ? a.n - r : rows;
        b.X += r * a.ld;
        b.labels += r;
        b.keys += r;
        hipLaunchKernelGGL(k_screen_wide, dim3((unsigned)wide_blocks(b.n, b.k)), dim3(512), 4 * kWideStage, s, b);
        hipLaunchKernelGGL(k_screen_merge, dim3((unsigned)((b.n + 255) / 256)), dim3(256), 0, s, b);
        const hipError_t le = hipGetLastError();
        if (le != hipSuccess) return le;
    }
    return hipSuccess;
}

size_t screen_image_bytes(int k, int ld)
{
    const size_t nst = size_t(k + kScreenSC - 1) / kScreenSC;
    switch ((ld + 31) / 32) {
    case 1: return nst * ScreenGeom<1>::STAGE;
    case 2: return nst * ScreenGeom<2>::STAGE;
    case 3: return nst * ScreenGeom<3>::STAGE;
    default: return nst * ScreenGeom<4>::STAGE;
    }
}

hipError_t launch_screen(const ScreenArgs& a, int num_cu, hipStream_t s)
{
    if (a.n <= 0) return hipSuccess;
    switch ((a.ld + 31) / 32) {
    case 1: return launch_screen_nk<1>(a, num_cu, s);
    case 2: return launch_screen_nk<2>(a, num_cu, s);
    case 3: return launch_screen_nk<3>(a, num_cu, s);
    case 4: return launch_screen_nk<4>(a, num_cu, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace skm
