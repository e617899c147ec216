// sgq_quant.hip -- quantize / pack / unpack / dequantize kernels for gfx950.
//
// Bit-exactness contract with the reference quantizer (src/quantization.cpp):
//   max_abs  starts at 1e-8f and takes |x| only when |x| > max_abs, so NaN never
//            wins (:23-27, :57-61, :140-144).  A maximum is order-independent,
//            so the parallel reductions below give the serial loop's value.
//   scale    = max_abs / qmax and inv = qmax / max_abs, two correctly rounded
//            IEEE divisions (:29-30, :63-64, :146-147).
//   code     = max(lo, min(hi, round(x * inv))) with round half away from zero
//            and std::min/std::max operand order, so NaN gives hi (:36-37, :68-69, :151-152).
// Nothing in this file may be contracted into FMAs.
#include "sgq_internal.h"

#pragma clang fp contract(off)

namespace sgq {
namespace {

constexpr int kBlock = 256;

// Four floats at any 4-byte address.
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float ref_code(float x, float inv, float lo, float hi) {
    float v = roundf(x * inv);
    float m = (v < hi) ? v : hi;  // std::min(hi, v)
    return (lo < m) ? m : lo;     // std::max(lo, m)
}

__device__ __forceinline__ float ref_max(float m, float a) { return (a > m) ? a : m; }

__device__ __forceinline__ float wave_max(float m) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = ref_max(m, __shfl_xor(m, off));
    return m;
}

__device__ __forceinline__ bool valid_code(float v, float lo, float hi) {
    return v == truncf(v) && v >= lo && v <= hi;  // false for NaN and +-inf
}

__global__ void k_fill_zero(uint4* __restrict__ p, int64_t n16, unsigned char* __restrict__ tail, int ntail) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n16; i += stride) p[i] = make_uint4(0u, 0u, 0u, 0u);
    if (blockIdx.x == 0 && (int)threadIdx.x < ntail) tail[threadIdx.x] = 0;
}

__global__ void k_fill_bias(float* __restrict__ y, int64_t M, int64_t N, const float* __restrict__ bias) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < M * N; i += stride) y[i] = bias ? bias[i % N] : 0.0f;
}

// L lanes per group of G consecutive elements, V elements per load: a wavefront
// with 128-bit loads for long groups (rows of INT8 per channel), a wavefront
// for middle ones, eight lanes for groups of up to 128, where most of a
// wavefront would have nothing to load.
template <int L, int V>
__global__ void k_group_scales(const float* __restrict__ x, int64_t total, int64_t G, int64_t ngroups, float qmax,
                               float* __restrict__ scales, float* __restrict__ inv) {
    const int lane = threadIdx.x % L;
    const int64_t first = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / L;
    const int64_t step = ((int64_t)gridDim.x * blockDim.x) / L;
    for (int64_t g = first; g < ngroups; g += step) {
        const int64_t b = g * G;
        const int64_t e = (b + G < total) ? b + G : total;
        float m = 1e-8f;
        int64_t i = b;
        if constexpr (V == 4) {
            const int64_t n4 = (e - b) / 4;
#pragma unroll 4
            for (int64_t t = lane; t < n4; t += L) {
                const float4_u v = *(const float4_u*)(x + b + 4 * t);
                m = ref_max(ref_max(ref_max(ref_max(m, fabsf(v.x)), fabsf(v.y)), fabsf(v.z)), fabsf(v.w));
            }
            i += 4 * n4;
        }
#pragma unroll 4
        for (i += lane; i < e; i += L) m = ref_max(m, fabsf(x[i]));
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) m = ref_max(m, __shfl_xor(m, off));
        if (lane == 0) {
            scales[g] = m / qmax;
            if (inv) inv[g] = qmax / m;
        }
    }
}

__global__ void k_absmax_partial(const float* __restrict__ x, int64_t total, float* __restrict__ partial) {
    __shared__ float sm[kBlock / 64];
    float m = 1e-8f;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < total; i += stride) m = ref_max(m, fabsf(x[i]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = sm[0];
        for (int w = 1; w < kBlock / 64; ++w) r = ref_max(r, sm[w]);
        partial[blockIdx.x] = r;
    }
}

// Where a pack kernel's codes come from: x and the groups' scales found in the
// kernel, x and the inverse scales in inv, or fp32 codes (validated into *bad).
enum PackFrom { kFromX, kFromXInv, kFromCodes };

// The pack kernels take a tile of 32 rows by 128 columns per workgroup: x and
// the fp32 codes move in rows (512 contiguous bytes), the packed codes go
// through LDS so that a strip's rows leave as one 128-byte run (a thread per
// 16-byte chunk wrote chunks RQ * 16 bytes apart).  HBM bounds them.  Measured
// on MI355X in graphs, a quantize with fp32 codes, a thread per chunk and its
// passes -> this (us): INT4 4096 x 11008 g128 368 -> 82.5 (385 MB, 4.7 TB/s, what a
// large copy reaches), 4096 x 4096 g32 164 -> 28.1, g24 (scales found first) 184 ->
// 61, flat 4096 x 4100 g64 73.8 -> 43.8 (its scales by eight lanes a group); INT8
// 4096 x 4096 per tensor 125 -> 47.4, 4096 x 4097 per channel 124 -> 38.9.
constexpr int kPackRows = 32, kPackCols = 128;
// Tiles of one launch: a launch holds fewer than 2^32 threads, which the tiles
// of a very long, narrow weight exceed (K > 2^29 at up to 128 columns).
constexpr int64_t kPackTiles = (int64_t)1 << 22;

// INT8 strip-major: chunk (strip, row quad) is 4 columns x 4 rows, dword d
// column d, byte r row r.
template <PackFrom FROM>
__global__ __launch_bounds__(kBlock) void k_pack_i8_tiled(const float* __restrict__ src, uint32_t t0, int64_t K, int64_t N, int64_t RQ,
                                                          int64_t NS, int ncol, const float* __restrict__ inv,
                                                          int per_tensor, uint4* __restrict__ packed,
                                                          float* __restrict__ qdata, int* __restrict__ bad) {
    __shared__ __attribute__((aligned(16))) unsigned char col[kPackCols][kPackRows + 4];
    const uint32_t tile = t0 + blockIdx.x;
    const int64_t kb = tile / ncol, cb = tile - kb * ncol;
    const int64_t k0 = kb * kPackRows, n0 = cb * kPackCols;
    const int cq = threadIdx.x & 31, r0 = threadIdx.x >> 5;
    const int64_t n = n0 + 4 * cq;
    float v[4][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int64_t k = k0 + r0 + 8 * h;
        const float* p = src + k * N + n;
        if (k < K && n + 4 <= N) {
            const float4_u q = *(const float4_u*)p;
            v[h][0] = q.x, v[h][1] = q.y, v[h][2] = q.z, v[h][3] = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[h][e] = k < K && n + e < N ? p[e] : 0.0f;
        }
    }
    int badflag = 0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int r = r0 + 8 * h;
        const int64_t k = k0 + r;
        const float iv = FROM == kFromXInv && k < K ? (per_tensor ? inv[0] : inv[k]) : 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float c = 0.0f;
            if (k < K && n + e < N) {
                c = v[h][e];
                if constexpr (FROM == kFromCodes) {
                    if (!valid_code(c, -128.0f, 127.0f)) badflag = 1, c = 0.0f;
                } else {
                    c = ref_code(c, iv, -127.0f, 127.0f);
                }
            }
            v[h][e] = c;
            col[4 * cq + e][r] = (unsigned char)(int)c;
        }
        if (FROM == kFromXInv && qdata && k < K) {
            float* q = qdata + k * N + n;
            if (n + 4 <= N) {
                *(float4_u*)q = float4_u{v[h][0], v[h][1], v[h][2], v[h][3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) q[e] = v[h][e];
            }
        }
    }
    if (badflag) atomicOr(bad, 1);
    if (!packed) return;
    __syncthreads();
    // Chunk t % 8 of strip t / 8.
    const int64_t j = n0 / 4 + (threadIdx.x >> 3), rq = k0 / 4 + (threadIdx.x & 7);
    if (j < NS && rq < RQ) {
        uint32_t dw[4];
#pragma unroll
        for (int d = 0; d < 4; ++d)
            dw[d] = *(const uint32_t*)&col[4 * (threadIdx.x >> 3) + d][4 * (threadIdx.x & 7)];
        packed[j * RQ + rq] = make_uint4(dw[0], dw[1], dw[2], dw[3]);
    }
}

// A thread per chunk, consecutive threads on consecutive strips of the same rows:
// for weights that leave most of a 32 x 128 tile empty (launch_pack_i8_tiled).
template <PackFrom FROM>
__global__ __launch_bounds__(kBlock) void k_pack_i8_chunks(const float* __restrict__ src, int64_t K, int64_t N, int64_t RQ,
                                                           int64_t NS, int64_t nchunks, const float* __restrict__ inv,
                                                           int per_tensor, uint4* __restrict__ packed,
                                                           float* __restrict__ qdata, int* __restrict__ bad) {
    for (int64_t c = blockIdx.x * (int64_t)kBlock + threadIdx.x; c < nchunks; c += (int64_t)gridDim.x * kBlock) {
        const int64_t rq = c / NS, j = c - rq * NS;
        const int64_t k0 = rq * 4, n0 = j * 4;
        uint32_t dw[4];
        int badflag = 0;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const int64_t n = n0 + d;
            uint32_t word = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t k = k0 + r;
                float v = 0.0f;
                if (k < K && n < N) {
                    v = src[k * N + n];
                    if constexpr (FROM == kFromCodes) {
                        if (!valid_code(v, -128.0f, 127.0f)) badflag = 1, v = 0.0f;
                    } else {
                        v = ref_code(v, per_tensor ? inv[0] : inv[k], -127.0f, 127.0f);
                        if (qdata) qdata[k * N + n] = v;
                    }
                }
                word |= ((uint32_t)(int)v & 0xFFu) << (8 * r);
            }
            dw[d] = word;
        }
        if (packed) packed[j * RQ + rq] = make_uint4(dw[0], dw[1], dw[2], dw[3]);
        if (badflag) atomicOr(bad, 1);
    }
}

// INT4 strip-major: the strips, the k-octet copy and (kFromX) the scales in
// both layouts from one read of x.  A thread takes eight columns of two rows,
// one strip dword each; a strip's 32 rows are consecutive dwords, and the
// k-octet dwords are gathered from the tile in LDS: block (cb, kb), dword t is
// column 16 cb + (t & 15), rows 32 kb + 8 (t >> 4) .. + 7 in nibbles 0..7.
// kFromX needs whole groups in the tile's rows (G divides 128 and N): the
// group's maximum is taken over its G / 8 lanes.
template <PackFrom FROM>
__global__ __launch_bounds__(kBlock) void k_pack_i4_tiled(const float* __restrict__ src, uint32_t t0, int64_t K, int64_t N, int64_t G,
                                                          int64_t Kpad, int64_t RQ, int64_t NS, int ncol,
                                                          const float* __restrict__ inv, uint32_t* __restrict__ strips,
                                                          uint32_t* __restrict__ koct, int ngap,
                                                          float* __restrict__ scales, float* __restrict__ devscales,
                                                          float* __restrict__ qdata, int* __restrict__ bad) {
    constexpr int kOct = kPackCols / 8;
    __shared__ uint32_t word[kOct][kPackRows + 1];
    __shared__ float tsc[FROM == kFromX ? kOct : 1][kPackRows + 1];
    const uint32_t tile = t0 + blockIdx.x;
    const int64_t kb = tile / ncol, cb = tile - kb * ncol;
    const int64_t k0 = kb * kPackRows, j0 = cb * kOct;
    const int oc = threadIdx.x & (kOct - 1), r0 = threadIdx.x / kOct;
    const int64_t j = j0 + oc;
    float v[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t k = k0 + r0 + 16 * h;
        const bool in = k < K && j < NS;
        const float* p = src + k * N + 8 * j;
        const float4_u a = in ? *(const float4_u*)p : float4_u{0.f, 0.f, 0.f, 0.f};
        const float4_u c = in ? *(const float4_u*)(p + 4) : float4_u{0.f, 0.f, 0.f, 0.f};
        v[h][0] = a.x, v[h][1] = a.y, v[h][2] = a.z, v[h][3] = a.w;
        v[h][4] = c.x, v[h][5] = c.y, v[h][6] = c.z, v[h][7] = c.w;
    }
    int badflag = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = r0 + 16 * h;
        const int64_t k = k0 + r;
        const bool in = k < K && j < NS;
        const int64_t i0 = k * N + 8 * j;
        float iv = 0.0f;
        if constexpr (FROM == kFromX) {
            float m = 1e-8f;
#pragma unroll
            for (int e = 0; e < 8; ++e) m = ref_max(m, fabsf(v[h][e]));
            for (int o = 1; o < (int)(G >> 3); o <<= 1) m = ref_max(m, __shfl_xor(m, o));
            iv = 7.0f / m;
            const float sc = m / 7.0f;
            if (in && (oc & (int)((G >> 3) - 1)) == 0) scales[i0 / G] = sc;
            tsc[oc][r] = k < K ? sc : 0.0f;
        } else if constexpr (FROM == kFromXInv) {
            if (in) iv = inv[i0 / G];  // N and G are multiples of 8: one group per octet
        }
        uint32_t w = 0;
        if (in) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float c = v[h][e];
                if constexpr (FROM == kFromCodes) {
                    if (!valid_code(c, -8.0f, 7.0f)) badflag = 1, c = 0.0f;
                } else {
                    c = ref_code(c, iv, -8.0f, 7.0f);
                }
                v[h][e] = c;
                w |= ((uint32_t)(int)c & 0xFu) << (4 * e);
            }
            if (FROM != kFromCodes && qdata) {
                *(float4_u*)(qdata + i0) = float4_u{v[h][0], v[h][1], v[h][2], v[h][3]};
                *(float4_u*)(qdata + i0 + 4) = float4_u{v[h][4], v[h][5], v[h][6], v[h][7]};
            }
        }
        word[oc][r] = w;
    }
    if (badflag) atomicOr(bad, 1);
    __syncthreads();
    const int64_t KB = (Kpad + 31) / 32, NB = (NS + 1) / 2;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int t = threadIdx.x + h * kBlock;
        // Strip t / 32, row t % 32.
        const int64_t js = j0 + (t >> 5), k = k0 + (t & 31);
        if (js < NS && k < Kpad) strips[4 * js * RQ + k] = word[t >> 5][t & 31];
        // k-octet dword t % 64 of column block t / 64.
        const int c = t & 15, g = (t >> 4) & 3;
        const int64_t blk = j0 / 2 + (t >> 6);
        if (blk < NB) {
            uint32_t w = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                w |= ((word[2 * (t >> 6) + (c >> 3)][8 * g + i] >> (4 * (c & 7))) & 0xFu) << (4 * i);
            koct[(blk * KB + kb) * 64 + (t & 63)] = w;
        }
        if constexpr (FROM == kFromX) {
            // Scale column of the tile's strip t / 32 where that strip is its first.
            const int64_t sc = js * 8 / G;
            if (js < NS && k < Kpad && (js * 8) % G == 0) devscales[sc * Kpad + k] = tsc[t >> 5][t & 31];
        }
    }
    // The dwords between the strips and the copy, so that the whole buffer is a
    // function of the codes.
    if (tile == 0 && (int)threadIdx.x < ngap) koct[(int64_t)threadIdx.x - ngap] = 0u;
}

// INT4 flat pack: one thread per byte (elements 2b, 2b+1 of the flattened tensor).
__global__ void k_pack_i4_flat(const float* __restrict__ src, int from_codes, int64_t total, int64_t G,
                               const float* __restrict__ inv, unsigned char* __restrict__ packed,
                               float* __restrict__ qdata, int* __restrict__ bad) {
    for (int64_t b = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; 2 * b < total;
         b += (int64_t)gridDim.x * blockDim.x) {
    uint32_t byte = 0;
    int badflag = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t i = 2 * b + h;
        if (i >= total) break;
        float v;
        if (from_codes) {
            v = src[i];
            if (!valid_code(v, -8.0f, 7.0f)) {
                badflag = 1;
                v = 0.0f;
            }
        } else {
            v = ref_code(src[i], inv[i / G], -8.0f, 7.0f);
            if (qdata) qdata[i] = v;
        }
        byte |= ((uint32_t)(int)v & 0xFu) << (4 * h);
    }
    if (packed) packed[b] = (unsigned char)byte;
    if (badflag) atomicOr(bad, 1);
    }
}

// devscales[sc][k] = scale of the first strip of scale column sc in row k.
__global__ void k_devscales_i4(const float* __restrict__ scales, int64_t K, int64_t N, int64_t G, int64_t Kpad,
                               int64_t spc, int64_t nsc, float* __restrict__ devscales) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nsc * Kpad;
         i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t sc = i / Kpad, k = i - sc * Kpad;
    const int64_t n = sc * spc * 8;
    devscales[i] = (k < K && n < N) ? scales[(k * N + n) / G] : 0.0f;
    }
}

__global__ void k_unpack_i8_tiled(const uint4* __restrict__ packed, int64_t K, int64_t N, int64_t RQ,
                                  int64_t NS, int64_t nchunks, const float* __restrict__ scales, int per_tensor,
                                  float* __restrict__ out) {
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nchunks;
         c += (int64_t)gridDim.x * blockDim.x) {
    const int64_t rq = c / NS, j = c - rq * NS;  // strip fastest: coalesced writes of out
    const int64_t k0 = rq * 4;
    const int64_t n0 = j * 4;
    const uint4 w = packed[j * RQ + rq];
    const uint32_t dw[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const int64_t n = n0 + d;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t k = k0 + r;
            if (k < K && n < N) {
                const float q = (float)(int)(signed char)(dw[d] >> (8 * r));
                out[k * N + n] = scales ? q * (per_tensor ? scales[0] : scales[k]) : q;
            }
        }
    }
    }
}

__global__ void k_unpack_i4_tiled(const uint4* __restrict__ packed, int64_t K, int64_t N, int64_t G, int64_t RQ,
                                  int64_t NS, int64_t nchunks, const float* __restrict__ scales,
                                  float* __restrict__ out) {
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nchunks;
         c += (int64_t)gridDim.x * blockDim.x) {
    const int64_t rq = c / NS, j = c - rq * NS;  // strip fastest: coalesced writes of out
    const int64_t k0 = rq * 4;
    const int64_t n0 = j * 8;
    const uint4 w = packed[j * RQ + rq];
    const uint32_t dw[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t k = k0 + r;
        if (k >= K) continue;
        const int64_t i0 = k * N + n0;
        const float s = scales ? scales[i0 / G] : 1.0f;  // one group per strip row (N % 8 == 0, G % 8 == 0)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float q = (float)(((int)(dw[r] << (28 - 4 * e))) >> 28);
            out[i0 + e] = scales ? q * s : q;
        }
    }
    }
}

__global__ void k_unpack_i4_flat(const unsigned char* __restrict__ packed, int64_t total, int64_t G,
                                 const float* __restrict__ scales, float* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t byte = packed[i >> 1];
    const float q = (float)(((int)(byte << (28 - 4 * (int)(i & 1)))) >> 28);
    out[i] = scales ? q * scales[i / G] : q;
    }
}

__global__ void k_dequant_codes(const float* __restrict__ q, const float* __restrict__ scales, int64_t total,
                                int mode, int64_t div, float* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x)
        out[i] = q[i] * (mode == 0 ? scales[0] : scales[i / div]);
}

inline unsigned grid_for(int64_t n, int64_t cap = 1 << 16) {
    int64_t g = ceil_div(n, kBlock);
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned)g;
}

}  // namespace

hipError_t launch_fill_zero(void* p, int64_t bytes, hipStream_t s) {
    if (bytes <= 0) return hipSuccess;
    const int64_t n16 = bytes / 16;
    const int ntail = (int)(bytes - n16 * 16);
    k_fill_zero<<<grid_for(n16 > 0 ? n16 : 1, 4096), kBlock, 0, s>>>(
        (uint4*)p, n16, (unsigned char*)p + n16 * 16, ntail);
    return hipGetLastError();
}

hipError_t launch_fill_bias(float* y, int64_t M, int64_t N, const float* bias, hipStream_t s) {
    if (M * N <= 0) return hipSuccess;
    k_fill_bias<<<grid_for(M * N, 4096), kBlock, 0, s>>>(y, M, N, bias);
    return hipGetLastError();
}

hipError_t launch_group_scales(const float* x, int64_t total, int64_t G, int64_t ngroups, float qmax, float* scales,
                               float* inv, hipStream_t s) {
    if (ngroups <= 0) return hipSuccess;
    if (G >= 1024)
        k_group_scales<64, 4><<<grid_for(ngroups * 64), kBlock, 0, s>>>(x, total, G, ngroups, qmax, scales, inv);
    else if (G > 128)
        k_group_scales<64, 1><<<grid_for(ngroups * 64), kBlock, 0, s>>>(x, total, G, ngroups, qmax, scales, inv);
    else
        k_group_scales<8, 1><<<grid_for(ngroups * 8), kBlock, 0, s>>>(x, total, G, ngroups, qmax, scales, inv);
    return hipGetLastError();
}

int64_t absmax_partial_count(int64_t total) {
    int64_t n = ceil_div(total, kBlock * 16);
    if (n < 1) n = 1;
    if (n > 1024) n = 1024;
    return n;
}

hipError_t launch_absmax_partial(const float* x, int64_t total, float* partial, int64_t nparts, hipStream_t s) {
    k_absmax_partial<<<(unsigned)nparts, kBlock, 0, s>>>(x, total, partial);
    return hipGetLastError();
}

// Weights that leave most of every tile empty: one row, a column or two, and
// long ones of up to 4 (16) columns, whose tiles outnumber the chip.  Measured (us
// a quantize with fp32 codes, tiles -> chunks): 1 x 2^20 22.7 -> 17.7, 2^20 x 1 67 ->
// 11.8, 2^20 x 3 80 -> 34, 131072 x 8 18.8 -> 13.7, x 16 19.7 -> 16.1; the tiles keep
// 2 x 2^20 (25.1 against 28.0), 4096 x 3 (10.5, 11.4), 131072 x 24 (23.0, 23.7), 2^20
// x 8 (90, 107).
static bool pack_i8_by_chunks(int64_t K, int64_t N) {
    constexpr int64_t kLong = 1 << 16, kVeryLong = 1 << 19;
    return K == 1 || N <= 2 || (K >= kLong && (N <= 4 || (N <= 16 && K < kVeryLong)));
}

hipError_t launch_pack_i8_tiled(const float* src, bool from_codes, int64_t K, int64_t N, const float* inv,
                                bool per_tensor, void* packed, float* qdata, int* bad, hipStream_t s) {
    const I8Geom g(K, N);
    if (g.chunks() <= 0) return hipSuccess;
    if (pack_i8_by_chunks(K, N)) {
        const unsigned blocks = grid_for(g.chunks());
        if (from_codes)
            k_pack_i8_chunks<kFromCodes><<<blocks, kBlock, 0, s>>>(src, K, N, g.RQ, g.NS, g.chunks(), inv, per_tensor,
                                                                   (uint4*)packed, qdata, bad);
        else
            k_pack_i8_chunks<kFromXInv><<<blocks, kBlock, 0, s>>>(src, K, N, g.RQ, g.NS, g.chunks(), inv, per_tensor,
                                                                  (uint4*)packed, qdata, bad);
        return hipGetLastError();
    }
    const int64_t ncol = ceil_div(N, kPackCols), blocks = ceil_div(g.Kpad, kPackRows) * ncol;
    if (blocks >= (int64_t)1 << 31) return hipErrorInvalidValue;
    for (int64_t t0 = 0; t0 < blocks; t0 += kPackTiles) {
        const unsigned n = (unsigned)(blocks - t0 < kPackTiles ? blocks - t0 : kPackTiles);
        if (from_codes)
            k_pack_i8_tiled<kFromCodes><<<n, kBlock, 0, s>>>(src, (uint32_t)t0, K, N, g.RQ, g.NS, (int)ncol, inv,
                                                             per_tensor, (uint4*)packed, qdata, bad);
        else
            k_pack_i8_tiled<kFromXInv><<<n, kBlock, 0, s>>>(src, (uint32_t)t0, K, N, g.RQ, g.NS, (int)ncol, inv,
                                                            per_tensor, (uint4*)packed, qdata, bad);
    }
    return hipGetLastError();
}

bool pack_i4_finds_scales(const I4Geom& g) { return g.tiled && g.N % g.G == 0 && kPackCols % g.G == 0; }

hipError_t launch_pack_i4_tiled(const float* src, bool from_codes, int64_t K, int64_t N, int64_t G, const float* inv,
                                void* packed, float* scales, float* devscales, float* qdata, int* bad, hipStream_t s) {
    const I4Geom g(K, N, G);
    if (g.chunks() <= 0) return hipSuccess;
    const int64_t ncol = ceil_div(g.NS, kPackCols / 8), blocks = g.KB() * ncol;
    if (blocks >= (int64_t)1 << 31) return hipErrorInvalidValue;
    const int ngap = (int)((g.koct_off() - g.chunks() * 16) / 4);
    uint32_t* koct = (uint32_t*)((char*)packed + g.koct_off());
    if (!from_codes && !inv && !pack_i4_finds_scales(g)) return hipErrorInvalidValue;
    for (int64_t t0 = 0; t0 < blocks; t0 += kPackTiles) {
        const unsigned n = (unsigned)(blocks - t0 < kPackTiles ? blocks - t0 : kPackTiles);
#define SGQ_PACK_I4(FROM_)                                                                                        \
    k_pack_i4_tiled<FROM_><<<n, kBlock, 0, s>>>(src, (uint32_t)t0, K, N, g.G, g.Kpad, g.RQ, g.NS, (int)ncol, inv, \
                                                (uint32_t*)packed, koct, ngap, scales, devscales, qdata, bad)
        if (from_codes)
            SGQ_PACK_I4(kFromCodes);
        else if (inv)
            SGQ_PACK_I4(kFromXInv);
        else
            SGQ_PACK_I4(kFromX);
#undef SGQ_PACK_I4
    }
    return hipGetLastError();
}

hipError_t launch_pack_i4_flat(const float* src, bool from_codes, int64_t total, int64_t G, const float* inv,
                               void* packed, float* qdata, int* bad, hipStream_t s) {
    const int64_t nbytes = ceil_div(total, 2);
    if (nbytes <= 0) return hipSuccess;
    k_pack_i4_flat<<<grid_for(nbytes), kBlock, 0, s>>>(src, from_codes, total, G, inv, (unsigned char*)packed,
                                                       qdata, bad);
    return hipGetLastError();
}

hipError_t launch_devscales_i4(const float* scales, const I4Geom& g, float* devscales, hipStream_t s) {
    const int64_t n = g.devscale_count();
    if (n <= 0) return hipSuccess;
    k_devscales_i4<<<grid_for(n), kBlock, 0, s>>>(scales, g.K, g.N, g.G, g.Kpad, g.spc, g.nsc, devscales);
    return hipGetLastError();
}

hipError_t launch_unpack_i8_tiled(const void* packed, int64_t K, int64_t N, const float* scales, bool per_tensor,
                                  float* out, hipStream_t s) {
    I8Geom g(K, N);
    const int64_t nchunks = g.chunks();
    if (nchunks <= 0 || K * N <= 0) return hipSuccess;
    k_unpack_i8_tiled<<<grid_for(nchunks), kBlock, 0, s>>>((const uint4*)packed, K, N, g.RQ, g.NS, nchunks, scales,
                                                           per_tensor, out);
    return hipGetLastError();
}

hipError_t launch_unpack_i4_tiled(const void* packed, int64_t K, int64_t N, int64_t G, const float* scales,
                                  float* out, hipStream_t s) {
    I4Geom g(K, N, G);
    const int64_t nchunks = g.chunks();
    if (nchunks <= 0 || K * N <= 0) return hipSuccess;
    k_unpack_i4_tiled<<<grid_for(nchunks), kBlock, 0, s>>>((const uint4*)packed, K, N, g.G, g.RQ, g.NS, nchunks, scales,
                                                           out);
    return hipGetLastError();
}

hipError_t launch_unpack_i4_flat(const void* packed, int64_t total, int64_t G, const float* scales, float* out,
                                 hipStream_t s) {
    if (total <= 0) return hipSuccess;
    k_unpack_i4_flat<<<grid_for(total), kBlock, 0, s>>>((const unsigned char*)packed, total, G, scales, out);
    return hipGetLastError();
}

hipError_t launch_dequant_codes(const float* q, const float* scales, int64_t total, int mode, int64_t div, float* out,
                                hipStream_t s) {
    if (total <= 0) return hipSuccess;
    k_dequant_codes<<<grid_for(total), kBlock, 0, s>>>(q, scales, total, mode, div, out);
    return hipGetLastError();
}

}  // namespace sgq
