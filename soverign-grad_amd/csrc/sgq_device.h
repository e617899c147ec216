// sgq_device.h -- device helpers shared by the forward kernels of libsgq.so
// (buffer loads, code conversion, the three-term bf16 split).  Device-only;
// include from .hip files.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sgq_internal.h"

namespace sgq {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Byte B of w read as a signed int8 and converted to fp32: the compiler emits
// one v_cvt_f32_i32 with an SDWA sign-extended byte select.  For INT4, a byte
// holding a code in its high nibble and zero below reads as 16*q exactly.
// Plain C++ rather than inline asm: the hazard recognizer does not track
// registers written inside inline asm, so an instruction that reads such a
// register too soon after it is written (an MFMA operand, for one) would get
// no wait states.
template <int B>
__device__ __forceinline__ float cvt_sbyte(uint32_t w) {
    return (float)(signed char)(w >> (8 * B));
}

__device__ __forceinline__ float i8_byte(uint32_t w, int b) {
    return b == 0 ? cvt_sbyte<0>(w) : (b == 1 ? cvt_sbyte<1>(w) : (b == 2 ? cvt_sbyte<2>(w) : cvt_sbyte<3>(w)));
}

__device__ __forceinline__ float f4get(const float4& v, int i) {
    return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}

// Raw buffer resource over [p, p + bytes): loads through it take a 32-bit
// lane offset plus a wave-uniform SGPR offset (no per-load 64-bit address
// math), and every dword past `bytes` reads as 0 -- which is how rows past K
// and row quads past the strip end contribute nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

constexpr int kOobOff = 0x40000000;  // a lane offset past every buffer the forward kernels read

__device__ __forceinline__ uint4 buf_load16(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_uint4(v.x, v.y, v.z, v.w);
}

// Loads of weight codes that a launch reads once (the GEMV with one row
// group, the INT4 skinny kernels: their workgroups partition the columns and
// K ranges) carry the non-temporal cache policy (`nt`): the stream does not
// displace x and the scales, which every workgroup of a scale column reads
// again.  Kernels whose workgroups read a code again (row groups, GEMM row
// tiles) keep the default policy.  Measured on MI355X (INT4
// g128, M = 1, graphs of 100 calls): 4096->4096 4.42 -> 4.03 us, 4096->11008
// 7.33 -> 6.85, 11008->4096 8.15 -> 7.26, 8192->8192 9.75 -> 8.27.
constexpr int kStreamPolicy = 2;  // buffer-instruction cache policy bit nt (gfx940+)
__device__ __forceinline__ uint4 buf_load16_stream(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kStreamPolicy);
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint32_t buf_load4_stream(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, kStreamPolicy);
}

// Four floats at byte offset voff + soff from any 4-byte address (128-bit
// buffer loads need dword alignment only); each float past the end is zero on
// its own (the range check of a raw buffer is by dword), so rows of any length
// and alignment load this way.
__device__ __forceinline__ float4 buf_load4f(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}

// silu(v) = v / (1 + exp(-v)), as simd::vec_silu (simd.hpp:103-108); the
// device expf differs from libm's by at most a few ulp, the division is
// correctly rounded.
__device__ __forceinline__ float silu_f32(float v) { return v / (1.0f + expf(-v)); }

// GemmEpilogue of one product (its bias added).
__device__ __forceinline__ float gemm_epilogue(const GemmEpilogue& e, float v, int64_t o) {
    if (e.gate) v = silu_f32(e.gate[o]) * v;
    if (e.res) v = v + e.res[o];
    return v;
}

// Workgroups are dispatched round-robin over the device's X = 2^xlog XCDs
// (workgroup b runs on XCD b % X; a full MI355X has 8, its partitions 4, 2 or
// 1, read per device as device_xcds), and each XCD has its own L2.  Strips
// that share a scale column (and, for the MFMA GEMM, tiles that share
// operands) should run on the same XCD, so the first X*(n/X) workgroup ids are
// permuted to give XCD x the contiguous range [x*(n/X), (x+1)*(n/X)); the
// remaining ids map to themselves.  A bijection on [0, n) for any xlog (0: the
// identity), so the XCD count only affects speed.
__device__ __forceinline__ int xcd_swizzle(int b, int n, int xlog) {
    const int per = n >> xlog;
    const int sw = (b & ((1 << xlog) - 1)) * per + (b >> xlog);
    return b >= (per << xlog) ? b : sw;  // a select, not a branch, ahead of the first loads
}

// Workgroup barrier ordering LDS accesses only: waits for this wave's LDS
// operations, not for its global loads.  __syncthreads() is a release fence
// as well, and gfx950 counts loads and stores on one counter (vmcnt), so it
// waits for every load in flight -- prefetched data included.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
// Upper halves (bf16 bits) of two floats in one dword, lo in bits 0-15.
__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ float trunc_bf16(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }

// Eight nibble codes (k order, nibble 0 first) as the bf16 values 16q of a B
// operand: high nibbles masked in place and low nibbles shifted up read as
// signed bytes 16q, converted exactly.
__device__ __forceinline__ bf16x8 nibbles_bf16x16(uint32_t t) {
    const uint32_t hi = t & 0xF0F0F0F0u, lo = (t << 4) & 0xF0F0F0F0u;
    const uint4 b = make_uint4(pack_hi16(cvt_sbyte<0>(lo), cvt_sbyte<0>(hi)), pack_hi16(cvt_sbyte<1>(lo), cvt_sbyte<1>(hi)),
                               pack_hi16(cvt_sbyte<2>(lo), cvt_sbyte<2>(hi)), pack_hi16(cvt_sbyte<3>(lo), cvt_sbyte<3>(hi)));
    return __builtin_bit_cast(bf16x8, b);
}

// h + m + l keeps all 24 bits of v only while the lowest of them is no smaller
// than bf16's smallest subnormal, 2^-133, that is for |v| >= 2^-110.  Kernels that
// took over from fp32 products put s * kScaleUp (or x * kScaleUp) into x * s and
// take kScaleUp (and the 16 of the codes) back out of the sums: times 2^16 that
// holds for every normal fp32 product, and a smaller one loses no more than
// fp32's own subnormals would.  A product or sum that this carries past fp32's
// range comes out non-finite, and is then recomputed in k order.
constexpr float kScaleUp = 65536.0f;
constexpr float kScaleDown = 0.0625f / 65536.0f;

// Splits eight floats into the bf16 planes h, m, l (four dwords each).
__device__ __forceinline__ void split3(const float* v, uint4& h, uint4& m, uint4& l) {
    // No fma: fused with the multiply that made v (x * s), a - trunc(a)
    // would take the unrounded product, and h + m + l would miss v by up to
    // an ulp.
#pragma clang fp contract(off)
    uint32_t ph[4], pm[4], pl[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = v[2 * i], b = v[2 * i + 1];
        ph[i] = pack_hi16(a, b);
        const float ra = a - trunc_bf16(a), rb = b - trunc_bf16(b);
        pm[i] = pack_hi16(ra, rb);
        pl[i] = pack_hi16(ra - trunc_bf16(ra), rb - trunc_bf16(rb));
    }
    h = make_uint4(ph[0], ph[1], ph[2], ph[3]);
    m = make_uint4(pm[0], pm[1], pm[2], pm[3]);
    l = make_uint4(pl[0], pl[1], pl[2], pl[3]);
}

// split3 of four floats (two dwords per plane).
__device__ __forceinline__ void split3_4(const float* v, uint2& h, uint2& m, uint2& l) {
#pragma clang fp contract(off)
    uint32_t ph[2], pm[2], pl[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float a = v[2 * i], b = v[2 * i + 1];
        ph[i] = pack_hi16(a, b);
        const float ra = a - trunc_bf16(a), rb = b - trunc_bf16(b);
        pm[i] = pack_hi16(ra, rb);
        pl[i] = pack_hi16(ra - trunc_bf16(ra), rb - trunc_bf16(rb));
    }
    h = make_uint2(ph[0], ph[1]);
    m = make_uint2(pm[0], pm[1]);
    l = make_uint2(pl[0], pl[1]);
}

// C neighbouring outputs of a row as the reference forms them (the non-finite
// fallback): sums over k in [k0, k1) of x[k] * (q[k][n + c] * s), in k order.
// C > 1: n .. n + C - 1 lie in one strip.  The loads of
// U k are issued together, and a thread stops once all its sums are NaN, which
// no further term changes: the NaN rows of a batch's inactive sequences end with
// their first k.  Measured (us, one k at a time to the end -> this): 256 x 2048 ->
// 5632 g32 with one row of NaN 323 -> 52, with one infinity 323 -> 104; a block
// step with inactive sequences, two of 8 at g128 350 -> 41, four of 24 at g32 481
// -> 72.
constexpr int kExactK = 8;
template <int BITS, int C, int U>
__device__ __forceinline__ void outputs_exact(const float* xrow, const uint4* W, const float* S, int mode, int Kpad, int RQ,
                                              int n, int k0, int k1, float (&acc)[C]) {
    const uint32_t* wd = reinterpret_cast<const uint32_t*>(W + (int64_t)(BITS == 8 ? n >> 2 : n >> 3) * RQ);
    if constexpr (BITS == 4) S += (int64_t)((n >> 3) / mode) * Kpad;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = 0.0f;
#pragma unroll 1
    for (int kb = k0; kb < k1; kb += U) {
        float xv[U], sv[U];
        uint32_t d[U][BITS == 8 ? C : 1];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int k = min(kb + i, k1 - 1);
            xv[i] = xrow[k];
            sv[i] = BITS == 8 && mode ? S[0] : S[k];
            if constexpr (BITS == 4) {
                d[i][0] = wd[k];
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c)
                    d[i][c] = reinterpret_cast<const unsigned char*>(wd)[(k >> 2) * 16 + ((n & 3) + c) * 4 + (k & 3)];
            }
        }
        bool all_nan = true;
#pragma unroll
        for (int c = 0; c < C; ++c) {
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const float q = BITS == 8 ? (float)(signed char)d[i][BITS == 8 ? c : 0]
                                          : (float)(((int)(d[i][0] << (28 - 4 * ((n & 7) + c)))) >> 28);
                if (kb + i < k1) acc[c] = fmaf(xv[i], q * sv[i], acc[c]);
            }
            all_nan = all_nan && isnan(acc[c]);
        }
        if (all_nan) break;
    }
}
// One INT8 output, one k at a time to the end: k_gemm3 inlines it for each of a
// thread's outputs, where anything longer costs its small batches (24 x 4096 ->
// 11008 24.2 -> 25.1 us).
__device__ __forceinline__ float output_exact_i8(const float* xrow, const uint4* W, const float* S, bool per_tensor, int RQ, int n, int k0,
                                 int k1) {
    float acc = 0.0f;
    for (int k = k0; k < k1; ++k) {
        const float q = (float)reinterpret_cast<const signed char*>(W)[((int64_t)(n >> 2) * RQ + (k >> 2)) * 16 +
                                                                       (n & 3) * 4 + (k & 3)];
        acc = fmaf(xrow[k], q * (per_tensor ? S[0] : S[k]), acc);
    }
    return acc;
}

}  // namespace
}  // namespace sgq
