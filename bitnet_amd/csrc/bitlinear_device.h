// Device arithmetic shared by the kernels: bf16 conversions, wave reductions, the RMSNorm, the
// squared-ReLU gate and the absmax quantizer on packed vectors.  One definition, so that kernels that
// compute the same step give the same bits.
#ifndef BITNET_AMD_BITLINEAR_DEVICE_H
#define BITNET_AMD_BITLINEAR_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

// fp32 -> bf16, round to nearest even: gfx950 has the conversion in hardware
// (two values per instruction)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f32x2_to_bf16x2(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) { return (uint16_t)(f32x2_to_bf16x2(f, 0.0f) & 0xffffu); }

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits
// for every outstanding global load of the wave, which would serialise the
// weight stream behind the barrier; here the weight words stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Wave-wide reductions with DPP lane permutes (no LDS): two quad permutes and
// two mirrors leave every lane of a 16-lane row with the row's result; the
// four row results are then combined through scalar registers.
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, (uint32_t)dpp_move<0xB1>((int)v));   // quad_perm [1,0,3,2]
    v = max(v, (uint32_t)dpp_move<0x4E>((int)v));   // quad_perm [2,3,0,1]
    v = max(v, (uint32_t)dpp_move<0x141>((int)v));  // row_half_mirror
    v = max(v, (uint32_t)dpp_move<0x140>((int)v));  // row_mirror
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return max(max(a, b), max(c, d));
}
__device__ __forceinline__ int wave_sum_i32(int v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0x141>(v);
    v += dpp_move<0x140>(v);
    return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
           __builtin_amdgcn_readlane(v, 48);
}

// max |x| over 8 packed bf16 as a bit pattern (|x| as bf16 bits orders like the values): one
// and + one packed 16-bit max per pair
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t absmax_bits8(const uint4& v, uint32_t cur) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    u16x2_t m = {(unsigned short)0, (unsigned short)0};
#pragma unroll
    for (int i = 0; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, d[i] & 0x7fff7fffu));
    const uint32_t both = __builtin_bit_cast(uint32_t, m);
    return max(cur, max(both & 0xffffu, both >> 16));
}

// One value to its int8 code, left in the low byte of the result: the product
// x * s in fp32 (mode 1: rounded to bf16) + 1.5 * 2^23, which rounds to the
// nearest integer (ties to even, as rint does) and leaves that integer's two's
// complement in the low mantissa bits, clamped to [-128, 127] there (clamping
// after rounding equals rounding after clamping: the bounds are integers; a NaN
// becomes -128).  In mode 0 x and s are bf16 values, so their product is exact in
// fp32 and one fused operation gives the sum's bits (a decode step of one
// sequence 584 -> 580 us, of two 693 -> 687, of eight 858 -> 855).
template <int MODE>
__device__ __forceinline__ uint32_t quant_low_byte(uint32_t x_f32_bits, float s32) {
    constexpr float kRound = 12582912.0f;
    const float x = __uint_as_float(x_f32_bits);
    float t;
    if (MODE == 1)
        t = bf16_to_f32(f32_to_bf16_rne(x * s32)) + kRound;
    else
        t = __builtin_fmaf(x, s32, kRound);
    return __float_as_uint(__builtin_amdgcn_fmed3f(t, kRound - 128.0f, kRound + 127.0f));
}

template <int MODE>
__device__ __forceinline__ int quant_one(uint32_t bits16, float s32) {
    return (int)(quant_low_byte<MODE>(bits16 << 16, s32) & 0xffu);
}

template <int MODE>
__device__ __forceinline__ uint2 quant_vec8(const uint4& v, float s32) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    uint32_t p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = quant_low_byte<MODE>(d[i] << 16, s32);
        const uint32_t hi = quant_low_byte<MODE>(d[i] & 0xffff0000u, s32);
        p[i] = __builtin_amdgcn_perm(hi, lo, 0x0c0c0400u);  // bytes (lo.0, hi.0, 0, 0)
    }
    // (p0.0, p0.1, p1.0, p1.1)
    return make_uint2(__builtin_amdgcn_perm(p[1], p[0], 0x05040100u), __builtin_amdgcn_perm(p[3], p[2], 0x05040100u));
}

// Activation scale from the row's |x| maximum (as bf16 bits).  torch evaluates
// 127 / t as t.reciprocal() * 127: a reciprocal, then a multiply.  The value
// returned is exactly representable in bf16.
template <int MODE>
__device__ __forceinline__ float quant_scale(uint32_t amax_bits) {
    float amax = __uint_as_float(amax_bits << 16);
    if (MODE == 0) {
        const float r = 1.0f / fmaxf(amax, 1e-5f);
        return bf16_to_f32(f32_to_bf16_rne(r * 127.0f));
    }
    amax = fmaxf(amax, bf16_to_f32(f32_to_bf16_rne(1e-5f)));
    const float r = bf16_to_f32(f32_to_bf16_rne(1.0f / amax));
    return bf16_to_f32(f32_to_bf16_rne(r * 127.0f));
}

__device__ __forceinline__ double dpp_sum_f64_row(double v) {
    // adds v over each 16-lane row with the same four lane permutes as above, on both halves of the double
#define BITLINEAR_DPP64(CTRL)                                                                      \
    {                                                                                              \
        const long long bits = __double_as_longlong(v);                                            \
        const int lo = dpp_move<CTRL>((int)(bits & 0xffffffffll)), hi = dpp_move<CTRL>((int)(bits >> 32)); \
        v += __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);                        \
    }
    BITLINEAR_DPP64(0xB1)
    BITLINEAR_DPP64(0x4E)
    BITLINEAR_DPP64(0x141)
    BITLINEAR_DPP64(0x140)
#undef BITLINEAR_DPP64
    return v;
}
__device__ __forceinline__ double wave_sum_f64(double v) {
    v = dpp_sum_f64_row(v);
    double t = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const long long bits = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_readlane((int)(bits & 0xffffffffll), 16 * r);
        const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), 16 * r);
        t += __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
    }
    return t;
}

// 8 bf16 (as 4 dwords) -> sum of squares; every square of a bf16 is exact in
// fp32 and the fp64 sum of a few thousand of them is exact for any data whose
// magnitudes span less than 2^24, so the result does not depend on the order
// of the additions.
__device__ __forceinline__ double sumsq8(const uint4& v) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = __uint_as_float(d[i] << 16), hi = __uint_as_float(d[i] & 0xffff0000u);
        acc += (double)(lo * lo) + (double)(hi * hi);
    }
    return acc;
}

// y = bf16(x * rstd * g) on 8 packed bf16
__device__ __forceinline__ uint4 norm8(const uint4& v, const uint4& g, float rstd) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    const uint32_t w[4] = {g.x, g.y, g.z, g.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = __uint_as_float(d[i] << 16) * rstd * __uint_as_float(w[i] << 16);
        const float hi = __uint_as_float(d[i] & 0xffff0000u) * rstd * __uint_as_float(w[i] & 0xffff0000u);
        o[i] = f32x2_to_bf16x2(lo, hi);
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// h = bf16(bf16(relu(x1)^2) * x3) on 8 packed bf16
__device__ __forceinline__ uint4 glu8(const uint4& a, const uint4& b) {
    const uint32_t d[4] = {a.x, a.y, a.z, a.w};
    const uint32_t e[4] = {b.x, b.y, b.z, b.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float r0 = fmaxf(__uint_as_float(d[i] << 16), 0.0f), r1 = fmaxf(__uint_as_float(d[i] & 0xffff0000u), 0.0f);
        const uint32_t sq = f32x2_to_bf16x2(r0 * r0, r1 * r1);
        const float s0 = __uint_as_float(sq << 16), s1 = __uint_as_float(sq & 0xffff0000u);
        const float lo = s0 * __uint_as_float(e[i] << 16), hi = s1 * __uint_as_float(e[i] & 0xffff0000u);
        o[i] = f32x2_to_bf16x2(lo, hi);
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

}  // namespace

#endif
