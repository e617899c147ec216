// sgq_flat.hip -- INT4 forward over the flat layout (src/quantization.cpp:
// 199-206): weights whose width or group is not a multiple of eight, for
// example an output head over an odd vocabulary.  The codes are the flattened
// [K,N] tensor, two per byte, and element i has scale S[i / G], so neither a
// row nor a group starts at a byte or a multiple of anything.
//
// Every form multiplies x by the reference's own product code * scale in fp32.
#include "sgq_device.h"
#include "sgq_internal.h"
#include "sgq_lanes.h"

namespace sgq {
namespace {

// Eight consecutive elements of the flat tensor: two dwords around them and
// the one or two scales they have (G >= 8).
struct FlatOct {
    uint32_t lo, hi;
    float s0, s1;
    int shift;  // bits of lo ahead of the first element
    int cut;    // elements cut .. 7 have scale s1
};

struct FlatSrc {
    __amdgpu_buffer_rsrc_t rP, rS;
    uint32_t tail;  // the last, partial dword of the codes
    int ptail;      // its index
    FastDiv G;
    int group;

    __device__ FlatSrc(const void* P, int nbytes, const float* S, int ngroups, FastDiv Gd, int g) : G(Gd), group(g) {
        // Whole dwords only: the partial one at the end is read by bytes.
        rP = make_rsrc(P, (uint32_t)nbytes & ~3u);
        rS = make_rsrc(S, (uint32_t)ngroups * 4u);
        ptail = nbytes >> 2;
        tail = 0;
        const unsigned char* b = (const unsigned char*)P + 4 * (int64_t)ptail;
        for (int i = 0; i < (nbytes & 3); ++i) tail |= (uint32_t)b[i] << (8 * i);
    }
    __device__ __forceinline__ uint32_t dword(int i) const {
        const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(rP, i * 4, 0, 0);  // zero past the whole dwords
        return i == ptail ? tail : v;
    }
    // Elements i .. i + 7; those past the last group have code and scale zero.
    __device__ __forceinline__ FlatOct load(int i) const {
        FlatOct o;
        const int g = G.div(i);
        o.lo = dword(i >> 3);
        o.hi = dword((i >> 3) + 1);
        o.s0 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rS, g * 4, 0, 0));
        o.s1 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rS, g * 4 + 4, 0, 0));
        o.shift = 4 * (i & 7);
        o.cut = (g + 1) * group - i;
        return o;
    }
};

// The eight weights code * scale.
__device__ __forceinline__ void flat_weights(const FlatOct& o, float (&w)[8]) {
    const uint32_t d = (uint32_t)((((uint64_t)o.hi << 32) | o.lo) >> o.shift);
    const uint32_t hi = d & 0xF0F0F0F0u, lo = (d << 4) & 0xF0F0F0F0u;  // bytes 16 q
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float q = i8_byte((e & 1) ? hi : lo, e >> 1) * 0.0625f;  // exact
        w[e] = q * (e < o.cut ? o.s0 : o.s1);
    }
}

struct FlatArgs {
    const float* x;
    int M, K, N;
    const void* P;
    int nbytes;
    const float* S;
    int ngroups, group;
    FastDiv G;
    const float* bias;
    float* y;
    int xlog;  // log2 of the device's XCD count
};

// Batches of a few rows, or of narrow weights.  A workgroup of 16 wavefronts owns
// 8 LC columns over all of K for MT batch rows (blockIdx.y picks the rows): LC lanes take eight
// consecutive columns each, the other 64 / LC lanes of a wavefront and the
// wavefronts take rows k in turn, so a wavefront reads runs of 4 LC bytes and
// a workgroup's loads walk the tensor in order.  x goes through LDS as [k][m]
// (one or two 128-bit reads give a lane its MT values).  The sums are combined
// over the lanes, then over the wavefronts in wavefront order.
//
// VALU-bound at eight rows (61% of the cycles issue VALU work): eight codes
// cost about 47 instructions to unpack and scale and 8 MT to multiply.
// Measured on MI355X, 2048 -> 32001 g32, thread per output -> this (us): 729 ->
// 18.8 at one row, 718 -> 29.8 at 4, 734 -> 43.5 at 8, 1135 -> 69 at 16, 2065
// -> 136 at 32; 4096 -> 1001 at one row 904 -> 18.2.  Neighbouring workgroups on
// different XCDs (each fetching the lines they share) took 59 us at 8 rows;
// two batches of loads in flight spilled and took 74.
constexpr int kFlatWaves = 16;

template <int H, int O, int STOP>
__device__ __forceinline__ void halve(float* v, int lane, int& base) {
    if constexpr (O >= STOP) {
        constexpr int h = H / 2;
        const bool upper = (lane & O) != 0;
#pragma unroll
        for (int i = 0; i < h; ++i) {
            if constexpr (O >= 16) {
                v[i] = swap_add<O>(v[i], v[i + h]);
            } else {
                const float send = upper ? v[i] : v[i + h], keep = upper ? v[i + h] : v[i];
                v[i] = keep + xor_lane<O>(send, lane);
            }
        }
        if (upper) base += h;
        halve<h, O / 2, STOP>(v, lane, base);
    }
}

template <int MT, int LC>
__global__ __launch_bounds__(kFlatWaves * 64) void k_flat_rows(const FlatArgs a) {
    constexpr int KPW = 64 / LC;             // rows of K per wavefront and step
    constexpr int STEP = kFlatWaves * KPW;   // rows of K per step
    constexpr int U = 4;                     // steps of loads in flight
    constexpr int KC = MT >= 4 ? 16384 / MT : 4096;  // rows of x in LDS
    constexpr int V = 8 * MT;                // sums per lane
    constexpr int OUT = V * LC;              // outputs of the workgroup
    constexpr int LEFT = V / KPW;            // sums a lane holds after the lane reduction
    static_assert(KC % (STEP * U) == 0 && LEFT >= 1, "steps fill a chunk");
    constexpr int kLds = kFlatWaves * OUT > KC * MT ? kFlatWaves * OUT : KC * MT;
    __shared__ __attribute__((aligned(16))) float lds[kLds];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cl = lane % LC, kl = lane / LC;
    const int m0 = blockIdx.y * MT, M = min(MT, a.M - m0);
    const int K = a.K, N = a.N;
    // Neighbours in columns share the lines at their edges: one XCD's L2.
    const int n0 = xcd_swizzle(blockIdx.x, gridDim.x, a.xlog) * 8 * LC;
    const FlatSrc src(a.P, a.nbytes, a.S, a.ngroups, a.G, a.group);
    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.0f;
    const int kw = wave * KPW + kl, c0 = n0 + 8 * cl;
    // Rows past K read x, codes and scales as zero.
    auto load = [&](FlatOct (&o)[U], int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * STEP + kw;
            o[u] = src.load(k < K ? k * N + c0 : a.ngroups * a.group);
        }
    };
    auto compute = [&](const FlatOct (&o)[U], int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float w[8], xv[MT];
            flat_weights(o[u], w);
            const float* xk = lds + (s0 + u * STEP + kw) * MT;
            if constexpr (MT >= 4) {
#pragma unroll
                for (int m = 0; m < MT; m += 4) {
                    const float4 q = *(const float4*)(xk + m);
                    xv[m] = q.x, xv[m + 1] = q.y, xv[m + 2] = q.z, xv[m + 3] = q.w;
                }
            } else {
#pragma unroll
                for (int m = 0; m < MT; ++m) xv[m] = xk[m];
            }
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[m * 8 + e] = fmaf(xv[m], w[e], acc[m * 8 + e]);
        }
    };
    for (int kc = 0; kc < K; kc += KC) {
        const int rows = min(KC, (K - kc + STEP * U - 1) / (STEP * U) * (STEP * U));
        FlatOct o[U];
        load(o, kc);  // under the loads of x
        if (kc > 0) __syncthreads();
#pragma unroll
        for (int m = 0; m < MT; ++m)
            for (int k = threadIdx.x; k < rows; k += kFlatWaves * 64)
                lds[k * MT + m] = (m < M && kc + k < K) ? a.x[(int64_t)(m0 + m) * K + kc + k] : 0.0f;
        __syncthreads();
        for (int s0 = 0; s0 < rows; s0 += STEP * U) {
            if (s0 > 0) load(o, kc + s0);
            compute(o, s0);
        }
    }
    int base = 0;
    halve<V, 32, LC>(acc, lane, base);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LEFT; ++i) lds[wave * OUT + cl * V + base + i] = acc[i];
    __syncthreads();
    for (int t = threadIdx.x; t < OUT; t += kFlatWaves * 64) {
        // Output t: row t / (8 LC), column t % (8 LC) of the workgroup.
        const int m = t / (8 * LC), c = t % (8 * LC);
        const int at = (c >> 3) * V + m * 8 + (c & 7);
        float r = 0.0f;
#pragma unroll
        for (int w = 0; w < kFlatWaves; ++w) r += lds[w * OUT + at];
        const int n = n0 + c;
        if (m < M && n < N) a.y[(int64_t)(m0 + m) * N + n] = a.bias ? r + a.bias[n] : r;
    }
}

// Larger batches: 128 x 128 tiles on v_mfma_f32_16x16x4_f32, four wavefronts in
// 2 x 2, as k_gemm (sgq_linear.hip): 32 k per stage through LDS, A as [m][k], B
// dequantized as [n][k], one stage computed while the next is loaded.  The
// fp32 MFMA bounds it: 128 x 2048 -> 32001 takes 244 us (69 TFLOP/s), 7207 with
// a thread per output.
constexpr int kFT = 128, kFK = 32, kFStride = kFK + 4;

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_flat_gemm(const FlatArgs a) {
    __shared__ __attribute__((aligned(16))) float As[2][kFT][kFStride], Bs[2][kFT][kFStride];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1, lr = lane & 15;
    const int M = a.M, K = a.K, N = a.N;
    const int ntn = (N + kFT - 1) / kFT;
    const int tm = blockIdx.x / ntn, tn = blockIdx.x - tm * ntn;
    const int m0 = tm * kFT, n0 = tn * kFT;
    const int KT = (K + kFK - 1) / kFK;
    const FlatSrc src(a.P, a.nbytes, a.S, a.ngroups, a.G, a.group);
    const int mrows = min(kFT, M - m0);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(a.x + (int64_t)m0 * K, (uint32_t)mrows * (uint32_t)K * 4u);
    // A: thread t loads k t % 32 of rows t / 32 + 8 i (any K and alignment);
    // B: column octet t % 16 of rows k t / 16 and t / 16 + 16.
    float av[16];
    FlatOct bo[2];
    auto load = [&](int kt) {
        const int k = kt * kFK + (tid & 31);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            av[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                rX, k < K ? (((tid >> 5) + 8 * i) * K + k) * 4 : kOobOff, 0, 0));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int kb = kt * kFK + (tid >> 4) + 16 * h;
            bo[h] = src.load(kb < K ? kb * N + n0 + 8 * (tid & 15) : a.ngroups * a.group);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 16; ++i) As[buf][(tid >> 5) + 8 * i][tid & 31] = av[i];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float w[8];
            flat_weights(bo[h], w);
#pragma unroll
            for (int e = 0; e < 8; ++e) Bs[buf][8 * (tid & 15) + e][(tid >> 4) + 16 * h] = w[e];
        }
    };
    floatx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    load(0);
    store(0);
    __syncthreads();
    for (int kt = 0; kt < KT; ++kt) {
        const int buf = kt & 1;
        load(kt + 1);  // past the last stage: zeros, not stored
#pragma unroll
        for (int sb = 0; sb < kFK / 16; ++sb) {
            const int lk = sb * 16 + (lane >> 4) * 4;
            float4 av4[4], bv4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av4[i] = *(const float4*)&As[buf][wm * 64 + i * 16 + lr][lk];
#pragma unroll
            for (int j = 0; j < 4; ++j) bv4[j] = *(const float4*)&Bs[buf][wn * 64 + j * 16 + lr][lk];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f4get(av4[i], kk), f4get(bv4[j], kk),
                                                                         acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < KT) store(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + wn * 64 + j * 16 + lr;
            if (n >= N) continue;
            const float bv = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wm * 64 + i * 16 + (lane >> 4) * 4 + r;
                if (m < M) a.y[(int64_t)m * N + n] = a.bias ? acc[i][j][r] + bv : acc[i][j][r];
            }
        }
}

// ---------------------------------------------------------------------------
// A short K (flat_form), and the remaining flat weights: groups or widths below
// eight, codes at an odd address or past 32-bit indices or grids.  One thread per
// output; per-element scale index, the reference's own product code*scale, FMA
// accumulation in k order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_linear_i4_flat(const float* __restrict__ x, int64_t M, int64_t K,
                                                             int64_t N, const unsigned char* __restrict__ P,
                                                             const float* __restrict__ S, int64_t G,
                                                             const float* __restrict__ bias, float* __restrict__ y) {
    for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < M * N;
         o += (int64_t)gridDim.x * blockDim.x) {
        const int64_t m = o / N, n = o - m * N;
        float acc = 0.0f;
        for (int64_t k = 0; k < K; ++k) {
            const int64_t i = k * N + n;
            const uint32_t byte = P[i >> 1];
            const float q = (float)(((int)(byte << (28 - 4 * (int)(i & 1)))) >> 28);
            acc = fmaf(x[m * K + k], q * S[i / G], acc);
        }
        y[o] = bias ? acc + bias[n] : acc;
    }
}

// 128 columns per workgroup of the row form where that gives every CU one, else 64.
bool flat_wide(int64_t groups, int64_t N, int64_t cus) { return ceil_div(N, 128) * groups >= cus; }

// The form with the least expected time, us on an MI355X, fitted to nine hundred
// shapes of 1 to 65536 rows, K 1 to 4096 and N 9 to 32001 with each form timed: of
// those the choice is at most 9% slower than a thread per output, and all but ten
// lie within 15% of the best form (those ten take 10 to 30 us).
//  - a thread per output walks K at 0.17 us a step while the chip is not full,
//    then at 1.4 products per ps and 0.65 outputs per ps.  Short K: 100000 x 8 ->
//    12 12.4 us against 397 for the row form and 13 for tiles, 39 x 6 -> 9671 5.1
//    against 20, one row x 3 -> 7095 2.8 against 5.0.
//  - the row form: a workgroup per CU at a time, each a fixed cost (x into LDS, the
//    reductions) and a time per k, by rows and columns per workgroup.
//  - tiles cost 3.6 us for 32 k and every 128 rows, however few of them: 2048 ->
//    32001 takes the rows 34 us per eight and tiles 241 up to 128 rows.
enum class FlatForm { kThreads, kRows, kTiles };
FlatForm flat_form(int64_t M, int64_t K, int64_t N, int64_t cus) {
    const double k = (double)K, mn = (double)M * (double)N;
    FlatForm best = FlatForm::kThreads;
    double t = 3.0 + 0.17 * k + mn * (k / 1.4e6 + 1 / 6.5e5);
    const int mlog = M == 1 ? 0 : (M == 2 ? 1 : (M <= 4 ? 2 : 3));
    const int64_t groups = ceil_div(M, (int64_t)1 << mlog);
    if (groups <= 65535) {  // grid.y
        static const double fixed[2][4] = {{3.0, 3.5, 4.5, 7.5}, {4.5, 6.5, 8.5, 9.0}};
        static const double per_k[2][4] = {{.003, .0033, .0045, .0065}, {.0055, .007, .0085, .0135}};
        const bool wide = flat_wide(groups, N, cus);
        const int64_t rounds = ceil_div(groups * ceil_div(N, wide ? 128 : 64), cus);
        const double rows = 3.0 + (wide && rounds == 1 && mlog == 3 ? 6.0 : 0.0) +
                            (double)rounds * (fixed[wide][mlog] + per_k[wide][mlog] * k);
        if (rows < t) t = rows, best = FlatForm::kRows;
    }
    if (M > 32) {
        const int64_t tiles = ceil_div(M, kFT) * ceil_div(N, kFT);
        const double gemm =
            12.0 + mn / 5.5e5 + (double)ceil_div(K, kFK) * (tiles <= cus ? 3.6 : 2.9 * (double)ceil_div(tiles, cus));
        if (gemm < t) best = FlatForm::kTiles;
    }
    return best;
}

template <int MT>
void flat_rows_launch(const FlatArgs& a, int64_t cus, hipStream_t s) {
    const unsigned groups = (unsigned)ceil_div(a.M, MT);
    if (flat_wide(groups, a.N, cus))
        k_flat_rows<MT, 16><<<dim3((unsigned)ceil_div(a.N, 128), groups), kFlatWaves * 64, 0, s>>>(a);
    else
        k_flat_rows<MT, 8><<<dim3((unsigned)ceil_div(a.N, 64), groups), kFlatWaves * 64, 0, s>>>(a);
}

}  // namespace

hipError_t launch_linear_i4_flat(const float* x, int64_t M, int64_t K, int64_t N, const void* packed,
                                 const float* scales, int64_t G, const float* bias, float* y, hipStream_t s) {
    // Elements are indexed in 31 bits, one row and a workgroup's columns past
    // the last; an octet has at most two scales from groups of eight on; codes
    // are read by aligned dwords.  Rows fit an int, and a grid of 64 columns to
    // 1024 threads stays below 2^32 threads.
    const bool fast = G >= 8 && N >= 8 && G < ((int64_t)1 << 31) && (K + 1) * N + G + 1024 < ((int64_t)1 << 31) &&
                      K <= ((int64_t)1 << 21) && N < ((int64_t)1 << 27) && M < ((int64_t)1 << 31) &&
                      (((uintptr_t)packed) & 3) == 0;
    const int64_t cus = device_cus(s);
    const FlatForm form = fast ? flat_form(M, K, N, cus) : FlatForm::kThreads;
    if (form == FlatForm::kThreads) {
        int64_t blocks = ceil_div(M * N, 256);
        if (blocks > 65536) blocks = 65536;
        if (blocks < 1) blocks = 1;
        k_linear_i4_flat<<<(unsigned)blocks, 256, 0, s>>>(x, M, K, N, (const unsigned char*)packed, scales, G, bias, y);
        return hipGetLastError();
    }
    FlatArgs a{};
    a.x = x;
    a.M = (int)M, a.K = (int)K, a.N = (int)N;
    a.P = packed;
    a.nbytes = (int)ceil_div(K * N, 2);
    a.S = scales;
    a.ngroups = (int)ceil_div(K * N, G);
    a.group = (int)G;
    a.G = FastDiv((uint32_t)G);
    a.bias = bias;
    a.y = y;
    a.xlog = xcd_log2(device_xcds(s));
    if (form == FlatForm::kTiles)
        k_flat_gemm<<<(unsigned)(ceil_div(M, kFT) * ceil_div(N, kFT)), 256, 0, s>>>(a);
    else if (M == 1)
        flat_rows_launch<1>(a, cus, s);
    else if (M == 2)
        flat_rows_launch<2>(a, cus, s);
    else if (M <= 4)
        flat_rows_launch<4>(a, cus, s);
    else
        flat_rows_launch<8>(a, cus, s);
    return hipGetLastError();
}

}  // namespace sgq
