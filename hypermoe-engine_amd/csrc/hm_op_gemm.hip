// hm_op_gemm.hip -- the op-level products on the reference's [K x N]
// row-major weights (TensorBackend::matmul / matmulInt8Weights,
// CpuTensorBackend.cpp:87-190) on the matrix cores.
//
//   op_gemm_kernel<float, ..>   y = x W, FP32 matrix cores
//                               (v_mfma_f32_16x16x4_f32);
//   op_gemm_kernel<int8_t, ..>  y = s (x (q - zp)), bf16 matrix cores
//                               (v_mfma_f32_16x16x32_bf16): q - zp has at
//                               most eight significant bits, so it is exact
//                               in bf16, and 2^16 x is cut into three bf16
//                               parts that hold its 24 bits exactly (bf16
//                               ends at 2^-133: without the factor the last
//                               bits of x below 2^-110 would be lost); the
//                               three products of a term are exact and only
//                               their FP32 sums round.
//
// What bounds them: a call of the sizes an expert's rows have (1 to some
// hundred rows, K and N up to a few thousand) is 0.01 to 8 GFLOP on a few MB,
// so the time is set by how many compute units share it and by the loads'
// latency, not by the matrix rate.  A workgroup therefore takes a small tile
// (16 RF rows x 16 CF columns) over the whole K, its NW waves a K range each;
// they keep nothing in common until their sums meet in LDS, in wave order
// (no scratch memory, no second launch, the same bits on every run).
// Operands go straight to registers, D steps ahead: a lane's weight load
// is one vector of CF neighbouring columns of one K row, which gives it one
// value of each of the tile's CF column fragments (fragment f's column i is
// column CF i + f of the tile), so row-major weights need no transpose; its
// activation load is a run of its row's K, and the K order inside a step is
// permuted alike for both operands.
// What they measured stands at the rule that picks the tile, below.
#include "hm_device.h"

#include <limits.h>

#include <type_traits>

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
// vector loads from element-aligned addresses (odd K or N)
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32u __attribute__((aligned(1)));
typedef uint16_t u16u __attribute__((aligned(1)));

// ---- FP32 weights: a step is 16 K values; lane (g, i) = (lane / 16,
// lane % 16) holds K values 4 g .. 4 g + 3 of row i and of columns CF i ..,
// one per MFMA.
template <int RF, int CF>
struct StepF32 {
    static constexpr int K = 16;      // K values per step
    static constexpr int KL = 4;      // ... per lane
    f4 x[RF];
    float w[KL][CF];
};

// ---- INT8 weights: a step is 32 K values, eight per lane; w[j]: the CF
// columns' bytes of K value j.
template <int RF, int CF>
struct StepI8 {
    static constexpr int K = 32;
    static constexpr int KL = 8;
    f4 x[RF][2];
    uint32_t w[KL];
};

template <typename WT, int RF, int CF>
struct Step;
template <int RF, int CF>
struct Step<float, RF, CF> {
    typedef StepF32<RF, CF> type;
};
template <int RF, int CF>
struct Step<int8_t, RF, CF> {
    typedef StepI8<RF, CF> type;
};

// The upper halves of two floats as a pair of bf16.
__device__ __forceinline__ uint32_t op_high_halves(float lo, float hi) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo),
                                 0x07060302u);
}

// Eight floats as three bf16 vectors whose sum is exactly 2^16 x: each part the
// top 16 bits of what the parts before it leave (24 = 8 + 8 + 8 bits).  (A
// non-finite x gives NaN parts, as one of 2^112 and more does; such a tile
// is summed again on the FP32 instructions.)
constexpr float kOpScale = 0x1p16f;
__device__ __forceinline__ void op_split(const f4 (&x)[2], bf8 (&p)[3]) {
    uint32_t o[3][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        float a[2], b[2], c[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = kOpScale * x[h >> 1][2 * (h & 1) + e];
            a[e] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xffff0000u);
            const float r = v - a[e];
            b[e] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & 0xffff0000u);
            c[e] = r - b[e];
        }
        o[0][h] = op_high_halves(a[0], a[1]);
        o[1][h] = op_high_halves(b[0], b[1]);
        o[2][h] = op_high_halves(c[0], c[1]);
    }
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        uint4 v = make_uint4(o[l][0], o[l][1], o[l][2], o[l][3]);
        p[l] = __builtin_bit_cast(bf8, v);
    }
}

// x [M x K], w [K x N], y [M x N].  WT = int8_t: y = mant * (the sum of 2^16 x
// with p2-scaled weights), scale = 2^16 mant p2; zp the zero point; past: some
// (q - zp) * scale may be infinite.  WT = float: the last five arguments are not
// read.
template <typename WT, int RF, int CF, int NW, int D>
__global__ __launch_bounds__(64 * NW, NW == 16 ? 4 : 2) void op_gemm_kernel(
    const float* __restrict__ x, const WT* __restrict__ w, float* __restrict__ y, int64_t M,
    int64_t K, int64_t N, int64_t row_tiles, int64_t tiles, int32_t zp, float p2, float mant,
    float scale, bool past) {
    constexpr bool I8 = sizeof(WT) == 1;
    typedef typename Step<WT, RF, CF>::type S;
    constexpr int BM = 16 * RF, BN = 16 * CF;
    __shared__ float s_red[NW][BM][BN + 1];
    __shared__ int s_bad;  // the last tile (1, 2, ..) with an output that is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, li = lane & 15;
    const int64_t steps = (K + S::K - 1) / S::K;
    const int64_t s0 = wave * steps / NW, s1 = (wave + 1) * steps / NW;
    if (I8 && tid == 0) s_bad = 0;
    int round = 0;
    const float bias = I8 ? -(float)(128 + zp) * p2 : 0.0f;
    // Tiles are numbered column block major, row tile minor, in eight
    // contiguous ranges, one per XCD (workgroup i runs on XCD i % 8): the row
    // tiles of a column block meet in one XCD's L2, so each weight is fetched
    // once.
    const int64_t per = (tiles + 7) / 8;
    for (int64_t b = blockIdx.x; b < 8 * per; b += gridDim.x) {
        const int64_t tile = (b % 8) * per + b / 8;
        if (tile >= tiles || b / 8 >= per) continue;  // (uniform)
        const int64_t m0 = (tile % row_tiles) * BM, n0 = (tile / row_tiles) * BN;
        // Sources as a uniform base plus a 32-bit lane offset.  Rows past the
        // last repeat it; a lane's CF columns are one vector where N is a
        // multiple of CF (a vector past N repeats the last one) or the tile
        // is full.
        const float* xt = x + m0 * K;
        uint32_t xo[RF];
#pragma unroll
        for (int rf = 0; rf < RF; ++rf)
            xo[rf] = (uint32_t)(min((int64_t)(16 * rf + li), M - 1 - m0) * K + S::KL * g);
        const int64_t nv = n0 + CF * li;
        const uint32_t wo = (uint32_t)(S::KL * g * N + min(nv, N - CF) - n0);
        // full steps of whole vectors (offsets below 2^31 bytes); the others
        // one element at a time
        const bool vec = (N % CF == 0 || n0 + BN <= N) && N < (1 << 24) && K < (1 << 22);
        const int64_t sf = vec ? max(s0, min(s1, K / S::K)) : s0;

        auto load = [&](S& st, int64_t s) __attribute__((always_inline)) {
            const float* xs = xt + s * S::K;
            const WT* ws = w + s * S::K * N + n0;
#pragma unroll
            for (int rf = 0; rf < RF; ++rf) {
                if constexpr (I8) {
                    st.x[rf][0] = *reinterpret_cast<const f4u*>(xs + xo[rf]);
                    st.x[rf][1] = *reinterpret_cast<const f4u*>(xs + 4 + xo[rf]);
                } else {
                    st.x[rf] = *reinterpret_cast<const f4u*>(xs + xo[rf]);
                }
            }
#pragma unroll
            for (int j = 0; j < S::KL; ++j) {
                const WT* wp = ws + j * N;
                if constexpr (I8) {
                    if constexpr (CF == 4) st.w[j] = *reinterpret_cast<const u32u*>(wp + wo);
                    else st.w[j] = *reinterpret_cast<const u16u*>(wp + wo);
                } else if constexpr (CF == 4) {
                    const f4 v = *reinterpret_cast<const f4u*>(wp + wo);
#pragma unroll
                    for (int f = 0; f < CF; ++f) st.w[j][f] = v[f];
                } else {
                    const f2u v = *reinterpret_cast<const f2u*>(wp + wo);
                    st.w[j][0] = v[0];
                    st.w[j][1] = v[1];
                }
            }
        };
        // the last K step or a ragged column block: single elements from
        // clamped addresses; both operands are zero past K (a non-finite
        // element of the last row must not meet a zero)
        auto load_elements = [&](S& st, int64_t s) __attribute__((always_inline)) {
            const int64_t k = s * S::K + S::KL * g;
#pragma unroll
            for (int j = 0; j < S::KL; ++j) {
                const bool in = k + j < K;
                const int64_t kk = in ? k + j : K - 1;
#pragma unroll
                for (int rf = 0; rf < RF; ++rf) {
                    const float v = xt[min((int64_t)(16 * rf + li), M - 1 - m0) * K + kk];
                    if constexpr (I8) st.x[rf][j >> 2][j & 3] = in ? v : 0.0f;
                    else st.x[rf][j] = in ? v : 0.0f;
                }
                uint32_t packed = 0;
#pragma unroll
                for (int f = 0; f < CF; ++f) {
                    const WT v = w[kk * N + min(nv + f, N - 1)];
                    if constexpr (I8) packed |= (uint32_t)(uint8_t)(in ? v : (int8_t)zp) << (8 * f);
                    else st.w[j][f] = in ? v : 0.0f;
                }
                if constexpr (I8) st.w[j] = packed;
            }
        };

        f4 acc[RF][CF];
#pragma unroll
        for (int rf = 0; rf < RF; ++rf)
#pragma unroll
            for (int f = 0; f < CF; ++f) acc[rf][f] = f4{};
        auto multiply = [&](const S& st) __attribute__((always_inline)) {
            if constexpr (I8) {
                bf8 wb[CF];
#pragma unroll
                for (int f = 0; f < CF; ++f) {
                    uint32_t o[4];
#pragma unroll
                    for (int h = 0; h < 4; ++h) {
                        const uint32_t u0 = st.w[2 * h] ^ 0x80808080u, u1 = st.w[2 * h + 1] ^ 0x80808080u;
                        const float a = __builtin_fmaf((float)((u0 >> (8 * f)) & 255u), p2, bias);
                        const float b2 = __builtin_fmaf((float)((u1 >> (8 * f)) & 255u), p2, bias);
                        o[h] = op_high_halves(a, b2);
                    }
                    wb[f] = __builtin_bit_cast(bf8, make_uint4(o[0], o[1], o[2], o[3]));
                }
#pragma unroll
                for (int rf = 0; rf < RF; ++rf) {
                    bf8 xp[3];
                    op_split(st.x[rf], xp);
                    // the smallest parts first
#pragma unroll
                    for (int l = 2; l >= 0; --l)
#pragma unroll
                        for (int f = 0; f < CF; ++f)
                            acc[rf][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xp[l], wb[f], acc[rf][f], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int j = 0; j < S::KL; ++j)
#pragma unroll
                    for (int rf = 0; rf < RF; ++rf)
#pragma unroll
                        for (int f = 0; f < CF; ++f)
                            acc[rf][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.x[rf][j], st.w[j][f], acc[rf][f], 0, 0, 0);
            }
        };

        // the wave's whole steps, D loads ahead, then the others.  (INT8:
        // loads past the end repeat the last step and are not used; without
        // a branch around them the kernel holds its registers, 6.8 against
        // 8.4 us for one row.  FP32 has registers to spare: 10.5 against
        // 11.2 us with the branch.)
        if (s0 < sf) {
            S st[D];
#pragma unroll
            for (int d = 0; d < D; ++d)
                if (I8 || s0 + d < sf) load(st[d], min(s0 + d, sf - 1));  // (uniform)
#pragma clang loop unroll(disable)
            for (int64_t s = s0; s < sf; s += D) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    if (s + d < sf) multiply(st[d]);
                    if (I8 || s + d + D < sf) load(st[d], min(s + d + D, sf - 1));
                }
            }
        }
#pragma clang loop unroll(disable)
        for (int64_t s = sf; s < s1; ++s) {
            S st;
            load_elements(st, s);
            multiply(st);
        }
        // D of a 16 x 16 fragment: lane (g, i) holds rows 4 g .. 4 g + 3 of
        // column i.  AGAIN: only the outputs that are not finite yet, or all.
        ++round;
        auto finish = [&](auto again, bool all) __attribute__((always_inline)) {
            constexpr bool AGAIN = decltype(again)::value;
#pragma unroll
            for (int rf = 0; rf < RF; ++rf)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int f = 0; f < CF; ++f) s_red[wave][16 * rf + 4 * g + v][CF * li + f] = acc[rf][f][v];
            __syncthreads();
            bool bad = false;
            for (int u = tid; u < BM * BN; u += 64 * NW) {
                const int r = u / BN, c = u % BN;
                if (m0 + r >= M || n0 + c >= N) continue;
                float* out = y + (m0 + r) * N + n0 + c;
                if (AGAIN && !all && fabsf(*out) < __builtin_inff()) continue;
                float sum = s_red[0][r][c];
#pragma unroll
                for (int q = 1; q < NW; ++q) sum = __fadd_rn(sum, s_red[q][r][c]);
                if constexpr (I8 && !AGAIN) {
                    sum = __fmul_rn(sum, mant);
                    bad = bad || !(fabsf(sum) < __builtin_inff());
                }
                *out = sum;
            }
            if (I8 && !AGAIN && bad) s_bad = round;
            __syncthreads();  // the next sums go to s_red
        };
        finish(std::false_type{}, true);
        if constexpr (I8) {
            // An output is not finite (an activation that is not, or is 2^112 and
            // more, or a sum past the range): the tile again on the FP32
            // instructions, which give such outputs what their operands have, the
            // weights rounded as the reference rounds them (300 rows of K = 2048,
            // N = 768, all of it infinite: the call in 44 us, 17 where it is
            // finite, 444 with one lane's loop over K for each output); and every
            // tile where such weights may be infinite (past).
            if (s_bad != round && !past) continue;  // (uniform)
#pragma unroll
            for (int rf = 0; rf < RF; ++rf)
#pragma unroll
                for (int f = 0; f < CF; ++f) acc[rf][f] = f4{};
            const int64_t end = min(s1 * S::K, K);
#pragma clang loop unroll(disable)
            for (int64_t k0 = s0 * S::K; k0 < end; k0 += 4) {
                const int64_t k = min(k0 + g, K - 1);  // both operands are zero past K
                const bool in = k0 + g < K;
                float xv[RF];
#pragma unroll
                for (int rf = 0; rf < RF; ++rf) {
                    const float v = xt[min((int64_t)(16 * rf + li), M - 1 - m0) * K + k];
                    xv[rf] = in ? v : 0.0f;
                }
#pragma unroll
                for (int f = 0; f < CF; ++f) {
                    const int q = (int)w[k * N + min(nv + f, N - 1)] - zp;
                    const float wv = __fmul_rn((float)(in ? q : 0), scale);
#pragma unroll
                    for (int rf = 0; rf < RF; ++rf)
                        acc[rf][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[rf], wv, acc[rf][f], 0, 0, 0);
                }
            }
            finish(std::true_type{}, past);
        }
    }
}

// The tile of a product: the one whose rounds of workgroups over the compute
// units are expected to be the shortest.  A round of a tile takes about
// fixed + per_k K microseconds, measured alone on the chip at K = 768 and
// 2048 (1 to 150 rows).  So small calls get many small tiles (16 x 32: 1 to 16
// rows of K = 2048, N = 768 in 6.8 to 8.4 us INT8 and 10.5 to 11.2 us FP32)
// and large ones the tiles that read each operand least (32 x 64: 800 x 3072
// x 1536 in 50 us INT8 and 105 us FP32, where 16 x 32 takes 117 and 143).
// Against the kernels before these (a dot product per output and K part with
// a second launch adding the parts; 64 x 64 FMA tiles): 300 rows of K = 2048,
// N = 768 INT8 190 -> 11 us, 150 rows FP32 290 -> 12 us, one row INT8 22 + 4
// -> 7 us.
struct OpTile {
    int rf, cf;
    float fixed, per_k;
};
constexpr OpTile kOpTilesF32[] = {
    {1, 2, 3.2f, 3.7e-3f}, {1, 4, 4.0f, 5.6e-3f}, {2, 4, 4.0f, 9.0e-3f}, {4, 4, 4.8f, 15.5e-3f}};
constexpr OpTile kOpTilesI8[] = {
    {1, 2, 3.8f, 2.6e-3f}, {1, 4, 4.0f, 3.3e-3f}, {2, 4, 5.5f, 4.5e-3f}, {4, 4, 8.0f, 9.0e-3f}};

int op_gemm_tile(const OpTile (&tiles)[4], int64_t M, int64_t K, int64_t N) {
    int best = 0;
    double best_us = 0.0;
    for (int i = 0; i < 4; ++i) {
        const int64_t bm = 16 * tiles[i].rf, bn = 16 * tiles[i].cf;
        const double n = (double)((M + bm - 1) / bm) * (double)((N + bn - 1) / bn);
        const double us = std::ceil(n / 256.0) * (tiles[i].fixed + tiles[i].per_k * (double)K);
        if (i == 0 || us < best_us) {
            best = i;
            best_us = us;
        }
    }
    return best;
}

template <typename WT, int RF, int CF, int NW, int D>
int op_gemm_launch(const float* x, const WT* w, float* y, int64_t M, int64_t K, int64_t N,
                   int32_t zp, float p2, float mant, float scale, bool past, hipStream_t s) {
    const int64_t row_tiles = (M + 16 * RF - 1) / (16 * RF);
    const int64_t tiles = row_tiles * ((N + 16 * CF - 1) / (16 * CF));
    const int64_t want = (tiles + 7) / 8 * 8;
    hipLaunchKernelGGL((op_gemm_kernel<WT, RF, CF, NW, D>), dim3((unsigned)(want < (1 << 20) ? want : 1 << 20)),
                       dim3(64 * NW), 0, s, x, w, y, M, K, N, row_tiles, tiles, zp, p2, mant, scale, past);
    HM_LAUNCHED();
    return HM_OK;
}

}  // namespace

// y [M x N] = x [M x K] w [K x N], FP32.
int hm_launch_op_gemm_f32(const float* x, const float* w, float* y, int64_t M, int64_t K, int64_t N,
                          hipStream_t s) {
    switch (op_gemm_tile(kOpTilesF32, M, K, N)) {
    case 0: return op_gemm_launch<float, 1, 2, 16, 2>(x, w, y, M, K, N, 0, 1.0f, 1.0f, 1.0f, false, s);
    case 1: return op_gemm_launch<float, 1, 4, 8, 2>(x, w, y, M, K, N, 0, 1.0f, 1.0f, 1.0f, false, s);
    case 2: return op_gemm_launch<float, 2, 4, 4, 4>(x, w, y, M, K, N, 0, 1.0f, 1.0f, 1.0f, false, s);
    default: return op_gemm_launch<float, 4, 4, 4, 3>(x, w, y, M, K, N, 0, 1.0f, 1.0f, 1.0f, false, s);
    }
}

// y [M x N] = scale (x [M x K] (q [K x N] - zp)).  The power of two of the
// scale goes into the weights (q - zp times it is still exact in bf16) and
// its mantissa into the result, so that no sum is more than a factor of two
// from 2^16 times the result's own size.
int hm_launch_op_gemm_w8a32(const float* x, const int8_t* q, float scale, int32_t zp, float* y,
                            int64_t M, int64_t K, int64_t N, hipStream_t s) {
    int e;
    std::frexp(scale, &e);
    e = e - 1 < -100 ? -100 : e - 1 > 100 ? 100 : e - 1;
    const float p2 = std::ldexp(1.0f, e), mant = scale / p2 / kOpScale;
    // the reference's weights (q - zp) * scale may lie past the float range
    const bool past = std::isinf((float)std::max(127 - zp, 128 + zp) * scale);
    switch (op_gemm_tile(kOpTilesI8, M, K, N)) {
    case 0: return op_gemm_launch<int8_t, 1, 2, 16, 2>(x, q, y, M, K, N, zp, p2, mant, scale, past, s);
    case 1: return op_gemm_launch<int8_t, 1, 4, 8, 2>(x, q, y, M, K, N, zp, p2, mant, scale, past, s);
    case 2: return op_gemm_launch<int8_t, 2, 4, 4, 4>(x, q, y, M, K, N, zp, p2, mant, scale, past, s);
    default: return op_gemm_launch<int8_t, 4, 4, 4, 2>(x, q, y, M, K, N, zp, p2, mant, scale, past, s);
    }
}
