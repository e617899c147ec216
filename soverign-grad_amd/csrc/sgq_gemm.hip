// sgq_gemm.hip -- the INT4 prefill GEMM of the fused dequantize + matmul
// forward (src/quantization.cpp:189-206 for batches past the GEMV and skinny
// kernels), also INT8's where rows of x are not 16-byte aligned, and the sum of
// split-K partial results.
//
// k_gemm_wave runs the fp32 products on the bf16 matrix cores as three exact
// bf16 products each, as k_gemm3 does for INT8 (sgq_linear.hip): x * s split
// into three bf16 terms, codes exact in bf16, fp32 accumulation.  The terms hold
// all of a product from 2^-110 on (per tensor, of x), as in k_gemm3; groups
// below 128 ran on fp32 products before, and carry a factor of 2^16 that keeps
// all of fp32's normal range (kScaleUp; 0.5% of the time).
//
// Each wavefront computes a tile of its own, 16 RB rows by 128 columns, with
// no LDS and no barrier in the K loop.  The lanes load what their MFMA
// operands are made of straight from global memory: B operands are dwords of
// the k-octet copy, A operands the lane's eight x values (row lane & 15, k
// octet lane >> 4) times the scales of those k.  With A split in registers a
// wavefront can hold several scale columns: GPW groups of 128 / GPW columns
// split the same x values once per group, so groups of 32 and 64 run here too
// (the previous kernel needed one scale per 128-column tile, and smaller
// groups ran on the fp32 MFMA at a sixteenth of the bf16 rate).
//
// Why this shape: with the planes staged in LDS a 128 x 128 tile moved 96 KB
// through LDS per 32-k stage, as many cycles as its MFMAs take; here a stage
// is 96 MFMAs, 332 VALU instructions and 18 loads (RB = 4, one group), and
// the registers leave two wavefronts per SIMD.  In a stage the loads of the
// next are issued as soon as the registers they replace are consumed, and the
// split of the next row block (or the next stage's first) is interleaved with
// the MFMAs of the current one.
//
// What bounds it: the power limit.  At 2048 x 4096 -> 11008 (g128) the MFMAs
// run at 1.16 PFLOP/s (three times the 387 TFLOP/s of the product) with the
// clock at 1.9 GHz; a large bf16 library product on the same card runs at
// 1.2 PFLOP/s with the clock at 1.5-1.8 GHz.  Smaller groups are VALU-bound:
// the split costs 208 VALU instructions per group, row block set and stage.
// Measured on MI355X, both builds in turn, the kernels before this one -> this (us,
// with bias): g128 2048 x 4096 -> 11008 607 -> 473, 2048 x 11008 -> 4096 578 -> 439,
// 512 x 2048 -> 5632 74.9 -> 51.5; g64 512 x 2048 -> 5632 162 -> 58.1 to 60.5; g32 512
// x 2048 -> 5632 162 -> 72.1 to 74.8, 2048 x 4096 -> 11008 1684 -> 812, 40 x 11008 ->
// 4096 109 -> 37.5.  The error against 64 bits is no larger (g128 2048 x 4096 ->
// 11008 5.9e-7 -> 3.0e-7 with four K ranges, g32 512 x 2048 -> 5632 5.4e-7 -> 2.2e-7).
#include "sgq_device.h"
#include "sgq_internal.h"

namespace sgq {
namespace {

// Four floats at any 4-byte address, as 128-bit stores take them.
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kWaveCols = 128;  // columns of a wavefront's tile
constexpr int kWG = 256;        // threads per workgroup: four wavefronts
constexpr int kStageK = 32;     // k per stage: one 16x16x32 MFMA step
constexpr int64_t kMaxTiles = (int64_t)1 << 23;  // of a launch, which holds fewer than 2^32 threads

struct GemmWaveArgs {
    const float* x;
    int M, K, N;
    const uint4* W[3];  // weight blockIdx.y of one shape writes y + blockIdx.y * M * N
    const float* S[3];
    const float* bias[3];
    int spc, Kpad, RQ, NS;  // spc: strips per scale column
    int ko;                 // byte offset / 256 of the k-octet copy
    int KS, sps;            // K splits over workgroups, stages per split
    int sk;                 // K ranges within the workgroup: 1, 2 or 4
    GemmEpilogue ep;
    float* y;
    float* part;            // KS > 1: partial results of each weight, [KS][M][N]
    int ntn;                // workgroup tiles along N
    int xr, xlog;           // as k_gemm3: tile rows of an XCD's rectangle, log2 of the XCDs
};

// Workgroup b computes split b % KS (stages [kb0, kb1) of sps each) of tile
// b / KS; its four wavefronts are 4 / sk tiles of sk K ranges each.
template <int BITS, int RB, int GPW, bool PT>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_wave(const GemmWaveArgs a) {
    constexpr int CB = kWaveCols / 16;  // column blocks of 16 per wavefront
    constexpr int CPG = CB / GPW;       // of one scale group
    constexpr int BM = 16 * RB;
    constexpr int BW = BITS == 8 ? 2 : 1;  // code dwords per lane and column block
    __shared__ __attribute__((aligned(16))) float red[4][16][kWaveCols + 4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, g = lane >> 4;
    const int M = a.M, K = a.K, N = a.N, KS = a.KS, sk = a.sk;
    const int wi = blockIdx.y;
    const uint4* W = wi == 0 ? a.W[0] : (wi == 1 ? a.W[1] : a.W[2]);
    const float* S = wi == 0 ? a.S[0] : (wi == 1 ? a.S[1] : a.S[2]);
    const float* bias = wi == 0 ? a.bias[0] : (wi == 1 ? a.bias[1] : a.bias[2]);

    const int bsw = KS == 1 ? xcd_swizzle(blockIdx.x, gridDim.x, a.xlog) : (int)blockIdx.x;
    const int tile = bsw / KS, split = bsw - tile * KS;
    int tm = tile / a.ntn, tn = tile - tm * a.ntn;
    if (a.xr > 0) {
        const int per = (int)gridDim.x >> a.xlog, x = tile / per, l = tile - x * per;
        const int bw = per / a.xr, rects_m = (gridDim.x / a.ntn) / a.xr;
        tm = (x % rects_m) * a.xr + l % a.xr;
        tn = (x / rects_m) * bw + l / a.xr;
    }
    // Wavefront -> tile (and K range) within the workgroup.
    const int wtm = sk == 1 ? wave >> 1 : 0, wtn = sk == 4 ? 0 : wave & 1;
    const int kr = sk == 1 ? 0 : (sk == 2 ? wave >> 1 : wave);
    const int m0 = (tm * (sk == 1 ? 2 : 1) + wtm) * BM, n0 = (tn * (sk == 4 ? 1 : 2) + wtn) * kWaveCols;
    const int KT = (a.Kpad + kStageK - 1) / kStageK;
    const int kb0 = split * a.sps, kb1 = min(KT, kb0 + a.sps);
    const int per = (kb1 - kb0 + sk - 1) / sk;
    const int kt0 = min(kb1, kb0 + kr * per), kt1 = min(kb1, kt0 + per);
    const bool live = m0 < M && n0 < N;

    floatx4 acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    if (live && kt0 < kt1) {
        const int mrows = min(BM, M - m0);
        const __amdgpu_buffer_rsrc_t rX = make_rsrc(a.x + (int64_t)m0 * K, (uint32_t)mrows * (uint32_t)K * 4u);
        const int KB = (a.Kpad + 31) >> 5;
        // Column blocks (INT8: strips) past the weight's read as zero.
        __amdgpu_buffer_rsrc_t rW, rS[GPW];
        if constexpr (BITS == 8) {
            const int nstr = min(kWaveCols / 4, a.NS - n0 / 4);
            rW = make_rsrc(W + (int64_t)(n0 / 4) * a.RQ, (uint32_t)nstr * (uint32_t)a.RQ * 16u);
            rS[0] = make_rsrc(S, PT ? 4u : (uint32_t)K * 4u);
        } else {
            const int ncb = min(CB, (a.NS + 1) / 2 - n0 / 16);
            rW = make_rsrc(W + ((int64_t)a.ko + (int64_t)(n0 / 16) * KB) * 16, (uint32_t)ncb * (uint32_t)KB * 256u);
#pragma unroll
            for (int q = 0; q < GPW; ++q) {
                const int strip = min(n0 / 8 + q * (2 * CPG), a.NS - 1);
                rS[q] = make_rsrc(S + (int64_t)(strip / a.spc) * a.Kpad, (uint32_t)a.Kpad * 4u);
            }
        }
        int xo[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) xo[i] = ((i * 16 + lr) * K + 8 * g) * 4;

        uint32_t bw[CB][BW];
        float4 xq[RB][2], sv[GPW][2];
        // Past the last stage these read zeros, the next row or column block;
        // what they read is not used.
        auto loadB = [&](int kt) {
            if constexpr (BITS == 8) {
                // Column lr of block c is column 64 (c / 4) + 4 lr + c % 4 of the
                // tile: the four dwords of a chunk of strip lr serve four blocks.
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const uint4 w = buf_load16(rW, (lr * a.RQ + 2 * g + q) * 16, (16 * h * a.RQ + 8 * kt) * 16);
                        bw[4 * h][q] = w.x, bw[4 * h + 1][q] = w.y, bw[4 * h + 2][q] = w.z, bw[4 * h + 3][q] = w.w;
                    }
            } else {
#pragma unroll
                for (int c = 0; c < CB; ++c)
                    bw[c][0] = __builtin_amdgcn_raw_buffer_load_b32(rW, 4 * lane, (c * KB + kt) * 256, 0);
            }
        };
        auto loadS = [&](float4 (&s)[2], int q, int kt) {
            if constexpr (!PT) {
                s[0] = buf_load4f(rS[q], 32 * g, kt * 128);
                s[1] = buf_load4f(rS[q], 32 * g + 16, kt * 128);
            }
        };
        // Several scale groups: kScaleUp goes into the scales, or into x where
        // there are more groups than row blocks (fewer products per stage).
        constexpr bool kUpX = GPW > RB, kUpS = GPW > 1 && !kUpX;
        auto scaleUp = [&](float4 (&v)[2]) {
#pragma unroll
            for (int h = 0; h < 2; ++h) v[h].x *= kScaleUp, v[h].y *= kScaleUp, v[h].z *= kScaleUp, v[h].w *= kScaleUp;
        };
        // 128-bit buffer loads need dword alignment only, so rows of any K
        // (and any x) load the same way; full stages stay inside their row.
        auto loadX = [&](int i, int kt) {
            xq[i][0] = buf_load4f(rX, xo[i], kt * 128);
            xq[i][1] = buf_load4f(rX, xo[i] + 16, kt * 128);
        };
        bf16x8 bq[CB];
        auto convB = [&](int c) {
            if constexpr (BITS == 8) {
                // bytes of the column's dword in each row quad: k = 0..3, then 4..7
                const uint32_t lo = bw[c][0], hi = bw[c][1];
                bq[c] = __builtin_bit_cast(
                    bf16x8, make_uint4(pack_hi16(cvt_sbyte<0>(lo), cvt_sbyte<1>(lo)), pack_hi16(cvt_sbyte<2>(lo), cvt_sbyte<3>(lo)),
                                       pack_hi16(cvt_sbyte<0>(hi), cvt_sbyte<1>(hi)), pack_hi16(cvt_sbyte<2>(hi), cvt_sbyte<3>(hi))));
            } else {
                bq[c] = nibbles_bf16x16(bw[c][0]);
            }
        };
        // The planes of row block i scaled by s.
        auto split = [&](uint4 (&ap)[3], int i, const float4 (&s)[2]) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = PT ? f4get(xq[i][e >> 2], e & 3) : f4get(xq[i][e >> 2], e & 3) * f4get(s[e >> 2], e & 3);
            split3(v, ap[0], ap[1], ap[2]);
        };
        auto mfma = [&](const uint4& ap, int i, int c) {
            acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ap), bq[c], acc[i][c], 0, 0, 0);
        };
        const int kf = min(kt1, K / kStageK);  // full stages end here
        if (kt0 < kf) {
            uint4 ap[3];
            loadB(kt0);
#pragma unroll
            for (int q = 0; q < GPW; ++q) loadS(sv[q], q, kt0);
#pragma unroll
            for (int i = 0; i < RB; ++i) loadX(i, kt0);
#pragma unroll
            for (int c = 0; c < CB; ++c) convB(c);
            if constexpr (kUpS) scaleUp(sv[0]);
            if constexpr (kUpX) scaleUp(xq[0]);
            split(ap, 0, sv[0]);
            if (GPW == 1) loadX(0, kt0 + 1);
            for (int kt = kt0; kt < kf; ++kt) {
                loadB(kt + 1);
                float4 sn[2];  // one group: its next scales are needed before this stage's last use of the old ones
                if (GPW == 1) loadS(sn, 0, kt + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < GPW; ++q)
#pragma unroll
                    for (int i = 0; i < RB; ++i) {
                        const int i2 = (i + 1) % RB, q2 = i == RB - 1 ? (q + 1) % GPW : q;
                        const bool wrap = i2 == 0 && q2 == 0;
                        uint4 an[3];
                        // At the first use since they were loaded.
                        if (kUpS && i2 == 0) scaleUp(sv[q2]);
                        if (kUpX && q2 == 0) scaleUp(xq[i2]);
                        split(an, i2, GPW == 1 && wrap ? sn : sv[q2]);
                        if (i == RB - 1) {
#pragma unroll
                            for (int c = q * CPG; c < (q + 1) * CPG; c += 2) {
#pragma unroll
                                for (int p = 0; p < 3; ++p) {
                                    mfma(ap[p], i, c);
                                    mfma(ap[p], i, c + 1);
                                }
                                convB(c);
                                convB(c + 1);
                            }
                        } else {
#pragma unroll
                            for (int p = 0; p < 3; ++p)
#pragma unroll
                                for (int c = q * CPG; c < (q + 1) * CPG; ++c) mfma(ap[p], i, c);
                        }
                        if (q2 == GPW - 1) loadX(i2, wrap ? kt + 2 : kt + 1);
                        if (GPW > 1 && i2 == RB - 1) loadS(sv[q2], q2, kt + 1);
#pragma unroll
                        for (int p = 0; p < 3; ++p) ap[p] = an[p];
                        __builtin_amdgcn_sched_barrier(0);
                    }
                if (GPW == 1 && !PT) sv[0][0] = sn[0], sv[0][1] = sn[1];
            }
        }
        if (kf < kt1) {
            // The last, partial stage.  The scales and codes past K are zero or
            // unused; x past it is the next row's, so it is zeroed here.
            const int kt = kt1 - 1;
            const int k0 = kt * kStageK + 8 * g;
            loadB(kt);
#pragma unroll
            for (int q = 0; q < GPW; ++q) loadS(sv[q], q, kt);
#pragma unroll
            for (int i = 0; i < RB; ++i) loadX(i, kt);
            if constexpr (kUpS) {
#pragma unroll
                for (int q = 0; q < GPW; ++q) scaleUp(sv[q]);
            }
#pragma unroll
            for (int i = 0; i < RB; ++i) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    float4& v = xq[i][h];
                    const int left = K - k0 - 4 * h;
                    v.x = left > 0 ? v.x : 0.0f, v.y = left > 1 ? v.y : 0.0f;
                    v.z = left > 2 ? v.z : 0.0f, v.w = left > 3 ? v.w : 0.0f;
                }
                if constexpr (kUpX) scaleUp(xq[i]);
            }
#pragma unroll
            for (int c = 0; c < CB; ++c) convB(c);
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int q = 0; q < GPW; ++q) {
                    uint4 ap[3];
                    split(ap, i, sv[q]);
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int c = q * CPG; c < (q + 1) * CPG; ++c) mfma(ap[p], i, c);
                }
        }
    }

    // Sixteen rows at a time through LDS: the K ranges are added in range
    // order, and a row of a tile is stored by consecutive lanes.
    const int klo = kb0 * kStageK, khi = min(K, kb1 * kStageK);
    const float s_all = PT ? S[0] : 1.0f;
    const int nt = 4 / sk;  // tiles of the workgroup
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        if (i > 0) __syncthreads();
        if constexpr (BITS == 8) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    *(float4*)&red[wave][4 * g + r][64 * h + 4 * lr] =
                        make_float4(acc[i][4 * h][r], acc[i][4 * h + 1][r], acc[i][4 * h + 2][r], acc[i][4 * h + 3][r]);
        } else {
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[wave][4 * g + r][16 * j + lr] = acc[i][j][r];
        }
        __syncthreads();
        // A thread takes four columns at a time.
        for (int t = threadIdx.x; t < nt * 16 * (kWaveCols / 4); t += kWG) {
            const int tile_w = t / (4 * kWaveCols), row = (t / (kWaveCols / 4)) & 15, col = 4 * (t % (kWaveCols / 4));
            float4 v = *(const float4*)&red[tile_w][row][col];
            for (int q = 1; q < sk; ++q) {
                const float4 u = *(const float4*)&red[q * nt + tile_w][row][col];
                v.x += u.x, v.y += u.y, v.z += u.z, v.w += u.w;
            }
            const int um = sk == 1 ? tile_w >> 1 : 0, un = sk == 1 ? tile_w & 1 : tile_w;
            const int m = (tm * (sk == 1 ? 2 : 1) + um) * BM + i * 16 + row;
            const int n = (tn * (sk == 4 ? 1 : 2) + un) * kWaveCols + col;
            if (m >= M || n >= N) continue;
            // INT4 codes entered as 16q; per tensor, x itself in place of x * s.
            const float f = BITS == 8 ? s_all : (GPW > 1 ? kScaleDown : 0.0625f);
            v.x *= f, v.y *= f, v.z *= f, v.w *= f;
            // h + m + l turns an infinite x * s into inf - inf: recompute a
            // non-finite total as the reference's k-order sum.
            const int nc = BITS == 4 ? 4 : min(4, N - n);  // INT4: N is a multiple of 8
            if (!(isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w))) {
                float r[4];
                // (U for INT8: more loads together spill in the loop above.)
                outputs_exact<BITS, 4, BITS == 8 ? 2 : kExactK>(a.x + (int64_t)m * K, W, S, BITS == 8 ? (PT ? 1 : 0) : a.spc,
                                                                a.Kpad, a.RQ, n, klo, khi, r);
                v.x = isfinite(v.x) ? v.x : r[0], v.y = isfinite(v.y) ? v.y : r[1];
                v.z = isfinite(v.z) ? v.z : r[2], v.w = isfinite(v.w) ? v.w : r[3];
            }
            const int64_t o = (int64_t)m * N + n;
            float* out = KS > 1 ? a.part + (int64_t)(wi * KS + split) * M * N : a.y + (int64_t)wi * M * N;
            if (nc == 4) {
                if (KS == 1) {
                    if (bias) v.x += bias[n], v.y += bias[n + 1], v.z += bias[n + 2], v.w += bias[n + 3];
                    v.x = gemm_epilogue(a.ep, v.x, o), v.y = gemm_epilogue(a.ep, v.y, o + 1);
                    v.z = gemm_epilogue(a.ep, v.z, o + 2), v.w = gemm_epilogue(a.ep, v.w, o + 3);
                }
                *(f32x4_u*)(out + o) = f32x4_u{v.x, v.y, v.z, v.w};
            } else {
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    if (e >= nc) continue;
                    float w = f4get(v, e);
                    if (KS == 1) w = gemm_epilogue(a.ep, bias ? w + bias[n + e] : w, o + e);
                    out[o + e] = w;
                }
            }
        }
    }
}

// y = the epilogue of the sum over splits s = 0 .. KS-1, in that order, of
// part[s], plus the bias, for weight blockIdx.y.  V outputs per thread and load
// (V = 4: M * N a multiple of four, which keeps each partial result 16-byte
// aligned), every split's load issued before the first is added.  The leading
// scalar arguments are preloaded into SGPRs.
struct ReduceArgs {
    const float* bias[3];
    GemmEpilogue ep;
};
template <int V>
__global__ __launch_bounds__(kWG) void k_splitk_reduce(const float* __restrict__ part, float* y, int64_t MN, int KS,
                                                       int N, const ReduceArgs a) {
    const int wi = blockIdx.y;
    part += wi * KS * MN;
    const int64_t o = (blockIdx.x * (int64_t)kWG + threadIdx.x) * V;
    if (o >= MN) return;
    float t[kMaxSplits][V];
#pragma unroll
    for (int sp = 0; sp < kMaxSplits; ++sp) {
        if constexpr (V == 4) {
            const float4 q = sp < KS ? *(const float4*)(part + sp * MN + o) : make_float4(0.f, 0.f, 0.f, 0.f);
            t[sp][0] = q.x, t[sp][1] = q.y, t[sp][2] = q.z, t[sp][3] = q.w;
        } else {
            t[sp][0] = sp < KS ? part[sp * MN + o] : 0.0f;
        }
    }
    const float* bias = wi == 0 ? a.bias[0] : (wi == 1 ? a.bias[1] : a.bias[2]);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        float r = 0.0f;
#pragma unroll
        for (int sp = 0; sp < kMaxSplits; ++sp)
            if (sp < KS) r += t[sp][v];
        if (bias) r = r + bias[(o + v) % N];
        y[wi * MN + o + v] = gemm_epilogue(a.ep, r, o + v);
    }
}

}  // namespace

// Four row blocks where the 64-row tiles still give every SIMD a wavefront
// (each B operand serves more rows), two elsewhere and for several scale
// groups (VALU-bound, and the registers of four would spill).  Two K ranges
// where the grid already splits K, else four.  Measured (g128, us, two row
// blocks -> four): 2048 x 4096 -> 11008 484 -> 457 (1376 tiles x 1), 2048 x
// 4096 -> 4096 187 -> 176, 512 x 11008 -> 4096 141 -> 135; below the line 1024
// x 2048 -> 5632 78.6 against 80.5, 512 x 4096 -> 4096 70 against 71.  Four
// ranges against two without a split: 384 x 4096 -> 11008 116 against 134,
// 2048 x 4096 -> 11008 457 against 477; with one 40 x 4096 -> 4096 26.4
// against 23.5, 96 x 11008 -> 4096 45 against 43.
//
// A short K has too few stages for four ranges: a grid runs in rounds of two
// workgroups per CU, each costing its tiles' pass through LDS and its stages, and
// the arrangement with the least is taken, with two row blocks (their epilogue is
// shorter).  Fitted (us a round, four ranges / two / one): 6.2 / 8.5 / 12.6 and .44 /
// .97 / 1.98 a stage of 32 k.  Measured at K = 64 (us, the same, then the kernels
// before this one): g32 2048 rows -> 2048 19.9 / 14.4 / 16.3, 18.5; -> 4096 33.8 /
// 24.6 / 20.3, 24.2; -> 11008 81.7 / 57.2 / 48.2, 61.8; at K = 512 g128 4096 -> 16384
// 272 / 231 / 217, 271; at K = 96 512 rows -> 4096 11.1 / 13.2 / 17.0, 19.2.
GemmWaveShape gemm_wave_shape(int64_t M, int64_t K, int64_t N, bool one_scale, int KS, int64_t cus) {
    constexpr int64_t kShortK = 512;
    GemmWaveShape w;
    if (KS == 1 && K <= kShortK) {
        static const struct {
            int sk, round, stage;
        } forms[3] = {{4, 620, 44}, {2, 850, 97}, {1, 1260, 198}};
        int64_t best = 0;
        for (const auto& f : forms) {
            const GemmWaveShape t{2, f.sk};
            const int64_t rounds = ceil_div(ceil_div(M, t.rows()) * ceil_div(N, t.cols()), 2 * (cus < 1 ? 1 : cus));
            const int64_t cost = rounds * (f.round + f.stage * ceil_div(K, kStageK));
            if (best == 0 || cost < best) best = cost, w = t;
        }
        return w;
    }
    w.rb = one_scale && ceil_div(M, 64) * ceil_div(N, kWaveCols) * KS >= 4 * cus ? 4 : 2;
    w.sk = KS > 1 ? 2 : 4;
    return w;
}

hipError_t launch_gemm_wave(int bits, const float* x, int64_t M, int64_t K, int64_t N, int nw, const void* const* packed,
                            const float* const* scales, const float* const* bias, int mode, const GemmPlan& p,
                            const GemmWaveShape& w, const GemmEpilogue& ep, float* y, void* ws, hipStream_t s) {
    const int gpw = bits == 8 || mode % 16 == 0 ? 1 : (mode % 8 == 0 ? 2 : 4);
    if (!gemm_wave_takes(bits, mode) || (w.rb == 4 && gpw != 1) || nw < 1 || nw > 3 || (nw > 1 && (ep.gate || ep.res)))
        return hipErrorInvalidValue;
    const int64_t tm = ceil_div(M, w.rows()), tn = ceil_div(N, w.cols());
    if (p.KS == 1 && nw == 1 && tm > 1 && tm * tn >= kMaxTiles) {  // very many rows: two halves
        const int64_t h = tm / 2 * w.rows(), o = h * N;
        const GemmEpilogue rest{ep.gate ? ep.gate + o : nullptr, ep.res ? ep.res + o : nullptr};
        const hipError_t e = launch_gemm_wave(bits, x, h, K, N, 1, packed, scales, bias, mode, p, w, ep, y, ws, s);
        if (e != hipSuccess) return e;
        return launch_gemm_wave(bits, x + h * K, M - h, K, N, 1, packed, scales, bias, mode, p, w, rest, y + o, ws, s);
    }
    GemmWaveArgs a{};
    a.x = x;
    a.M = (int)M, a.K = (int)K, a.N = (int)N;
    for (int q = 0; q < nw; ++q) a.W[q] = (const uint4*)packed[q], a.S[q] = scales[q], a.bias[q] = bias[q];
    if (bits == 8) {
        const I8Geom g(K, N);
        a.Kpad = (int)g.Kpad, a.RQ = (int)g.RQ, a.NS = (int)g.NS;
    } else {
        const int64_t Kpad = round_up(K, kPadK);
        a.spc = mode;
        a.Kpad = (int)Kpad, a.RQ = (int)(Kpad / 4), a.NS = (int)(N / 8);
        a.ko = (int)(round_up(N / 8 * (Kpad / 4) * 16, 256) / 256);  // I4Geom::koct_off
    }
    a.KS = p.KS, a.sps = p.sps, a.sk = w.sk;
    a.ep = ep;
    a.y = y;
    a.part = p.KS > 1 ? (float*)ws : nullptr;
    a.ntn = (int)tn;
    const int xcds = device_xcds(s);
    a.xlog = xcd_log2(xcds);
    a.xr = p.KS == 1 ? xcd_rect_rows(tm, tn, w.rows() * K * 4, w.cols() * K * bits / 8, xcds) : 0;
    const dim3 grid((unsigned)(tm * tn * p.KS), (unsigned)nw);
#define SGQ_GEMM_WAVE(BITS_, GPW_, PT_)                              \
    if (w.rb == 4)                                                   \
        k_gemm_wave<BITS_, 4, GPW_, PT_><<<grid, kWG, 0, s>>>(a);    \
    else                                                             \
        k_gemm_wave<BITS_, 2, GPW_, PT_><<<grid, kWG, 0, s>>>(a)
    if (bits == 8 && mode) {
        SGQ_GEMM_WAVE(8, 1, true);
    } else if (bits == 8) {
        SGQ_GEMM_WAVE(8, 1, false);
    } else if (gpw == 1) {
        SGQ_GEMM_WAVE(4, 1, false);
    } else if (gpw == 2) {
        k_gemm_wave<4, 2, 2, false><<<grid, kWG, 0, s>>>(a);
    } else {
        k_gemm_wave<4, 2, 4, false><<<grid, kWG, 0, s>>>(a);
    }
#undef SGQ_GEMM_WAVE
    return hipGetLastError();
}

hipError_t launch_splitk_reduce(const float* part, int KS, int64_t M, int64_t N, int nw, const float* const* bias,
                                const GemmEpilogue& ep, float* y, hipStream_t s) {
    ReduceArgs a{};
    for (int w = 0; w < nw; ++w) a.bias[w] = bias[w];
    a.ep = ep;
    const int64_t MN = M * N;
    // Four outputs per thread only where that leaves every SIMD a few wavefronts.
    if (MN % 4 == 0 && MN >= (int64_t)1 << 20)
        k_splitk_reduce<4><<<dim3((unsigned)ceil_div(MN, 4 * kWG), (unsigned)nw), kWG, 0, s>>>(part, y, MN, KS, (int)N, a);
    else
        k_splitk_reduce<1><<<dim3((unsigned)ceil_div(MN, kWG), (unsigned)nw), kWG, 0, s>>>(part, y, MN, KS, (int)N, a);
    return hipGetLastError();
}

}  // namespace sgq
