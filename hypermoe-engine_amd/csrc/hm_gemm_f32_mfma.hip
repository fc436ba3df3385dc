// hm_gemm_f32_mfma.hip -- grouped FP32-weight expert GEMMs on the bf16 matrix
// cores (v_mfma_f32_16x16x32_bf16) for gfx950: the A5' path
// (ExpertExecutor.cpp:97-131 on CpuTensorBackend::matmul, :87-131).
//
// Every FP32 operand times 2^16 is cut into three bf16 parts of eight bits
// each, whose sum is it exactly (each the top 16 bits of what the parts before
// it leave; bf16 ends at 2^-133, so without the factor the last bits of
// operands below 2^-110 would be lost), and a product x w is the eight products
// of parts other than the two last ones': each exact, what is left out below
// 2^-32 |x w|, and the sums in FP32.  A single product is thus rounded once, as
// an FP32 matrix instruction rounds it (six products, without the second part
// times the third, leave out up to 2^-21 |x w|).  Long sums have a smaller error
// against 64-bit sums than those of FP32 matrix instructions on the whole values
// (an expert's output at K = 2048, 768: 4.6e-7 against 1.3e-6), as these round
// once per two k, the split ones' leading sums once per 32.  The reference sums
// each output sequentially in FP32: the results are within the FP32 path's 1e-3
// of it, not bit-identical (as the FMA tiles in hm_gemm.hip, which remain for
// other shapes).  An operand that is not finite gives NaN parts, one of 2^112 and
// more or a sum of 2^96 and more infinite ones; a tile with such a sum is
// summed again on FP32 matrix instructions (v_mfma_f32_16x16x4_f32), which give
// those outputs what their operands have (512 tokens, 8 experts top-2, H = 1024,
// I = 512, all of it NaN: the block in 165 us, 107 where it is finite, 4028 with
// one lane's loop over K for each output).
//
// What bounds them: reading the weights (1.2 GB at 64 experts: 230 us at a large
// copy's rate) once the matrix work fits under it.  FP32 MFMA does not (157
// TFLOP/s: 250 us for 512 tokens, 380 with its 64-row tiles' padding); eight bf16
// products take half of its cycles, and the cutting (6.5 vector instructions an
// element) somewhat more, beside them.  Measured at 512 tokens, 64 experts
// top-8: gate/up 410 -> 335 us, down 190 -> 161 us (six products: 296 and 146;
// eight of unscaled operands: 323 and 161).  With six products the cutting and
// the matrix work alone took 217 and 115 us, the loads alone 190 and 100, and
// what was left between was their overlap; cutting each activation once for all
// four waves (through LDS) halved the vector work and changed neither time.
//
// Workgroup: 4 waves, tile BM = 64 grouped rows x 128 weight rows (gate/up:
// 64 gate + the same 64 up columns; down: 128 output columns).  Wave c owns
// 32 of the weight rows (gate/up: 16 gate and the 16 up columns beside them)
// for every 16-row fragment that holds a row, so that a partial tile costs its
// fragments and no wave waits for another.  K moves in stages of 32 floats
// through a 2-slot LDS ring filled by 16-byte direct loads (global_load_lds), so
// that three workgroups fit a CU: they cover each other's waits better than a
// third slot does (gate/up, six products: 302 us; three slots, two workgroups
// 340).  Lane (g, i) = (lane/16, lane%16) supplies row or column i, k = 8 g ..
// 8 g + 7 of the stage.  Rows of a stage are 128 bytes; the 16-byte chunk c of
// row r is stored at slot c ^ (r % 8), which spreads a reader's rows over the LDS
// banks.  Tiles are numbered row tile major, column block minor, in eight
// contiguous ranges, one per XCD (workgroup i runs on XCD i % 8): the row tiles
// of one expert read its weights at about the same time from one L2.
#include "hm_device.h"
#include "hm_lds_dma.h"

#include <limits.h>

namespace {

constexpr int kFThreads = 256;
constexpr int kFBM = 64;            // grouped rows per tile
constexpr int kFRF = kFBM / 16;     // 16-row fragments
constexpr int kFBN = 128;           // weight rows per tile
constexpr int kFBK = 32;            // K floats per stage
constexpr int kFSlots = 2;
constexpr int kFRow = kFBK * 4;     // bytes per staged row
constexpr int kFStage = (kFBM + kFBN) * kFRow;  // 24 KB

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// Eight floats (two LDS chunks) times 2^16 as three bf16 vectors whose sum is
// exactly that.
constexpr float kFScale = 0x1p16f, kFUnscale = 0x1p-32f;
__device__ __forceinline__ void split_bf16(const f4& lo, const f4& hi, bf8 (&p)[3]) {
    uint32_t o[3][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        uint32_t a[2], b[2], c[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = kFScale * (h < 2 ? lo[2 * h + e] : hi[2 * (h - 2) + e]);
            a[e] = __builtin_bit_cast(uint32_t, v);
            const float r = v - __builtin_bit_cast(float, a[e] & 0xffff0000u);
            b[e] = __builtin_bit_cast(uint32_t, r);
            c[e] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, b[e] & 0xffff0000u));
        }
        o[0][h] = __builtin_amdgcn_perm(a[1], a[0], 0x07060302u);
        o[1][h] = __builtin_amdgcn_perm(b[1], b[0], 0x07060302u);
        o[2][h] = __builtin_amdgcn_perm(c[1], c[0], 0x07060302u);
    }
#pragma unroll
    for (int l = 0; l < 3; ++l) p[l] = __builtin_bit_cast(bf8, make_uint4(o[l][0], o[l][1], o[l][2], o[l][3]));
}

// Row tiles of every expert (ceil(count / kFBM)).  Every lane of the wave must
// be active.
__device__ __forceinline__ int64_t total_tiles(const int32_t* __restrict__ counts, int64_t experts) {
    int64_t n = 0;
    for (int64_t e = threadIdx.x & (HM_WAVE - 1); e < experts; e += HM_WAVE)
        n += ((int64_t)counts[e] + kFBM - 1) / kFBM;
#pragma unroll
    for (int d = 1; d < HM_WAVE; d <<= 1) n += __shfl_xor(n, d, HM_WAVE);
    return n;
}

// GATEUP: z[g, n] = silu(x_g . Wg[n]) * (x_g . Wu[n]), x_g = hidden[perm[g]],
// n in [0, I); tile columns n0 .. n0+63.  DOWN: y[g, n] = z_g . Wd[n],
// n in [0, H); tile columns n0 .. n0+127.  nbn: column blocks.
template <bool GATEUP>
__global__ __launch_bounds__(kFThreads, 3) void expert_f32_mfma_kernel(
    const float* __restrict__ x, int K, int N, int experts, const float* __restrict__ packed,
    int hidden, int inter, const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ perm_tokens, int nbn, float* __restrict__ out) {
    __shared__ __attribute__((aligned(1024))) char ring[kFSlots][kFStage];
    __shared__ int s_src[kFBM];
    __shared__ int s_bad;  // a sum of the tile is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the workgroup's tile (uniform, in scalar registers)
    const int total = __builtin_amdgcn_readfirstlane((int)total_tiles(counts, experts)) * nbn;
    const int per = (total + 7) / 8, idx = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= per || idx >= total) return;
    int64_t e64, mt64;
    if (!hm_locate_tile(counts, experts, kFBM, idx / nbn, &e64, &mt64)) return;
    const int e = __builtin_amdgcn_readfirstlane((int)e64), mt = __builtin_amdgcn_readfirstlane((int)mt64);
    const int64_t g0 = offsets[e] + (int64_t)mt * kFBM;
    const int rows = min(kFBM, counts[e] - mt * kFBM);
    const int64_t n0 = (int64_t)(idx % nbn) * (GATEUP ? kFBN / 2 : kFBN);
    if (tid == 0) s_bad = 0;
    if (tid < kFBM) {
        const int r = tid < rows ? tid : rows - 1;  // rows past the group repeat its last
        s_src[tid] = GATEUP ? perm_tokens[g0 + r] : (int)(g0 + r);
    }
    __syncthreads();
    // this wave's DMA rows: activation rows 16*wave .. +15 (2 loads, none
    // where the fragment holds no row), weight rows 32*wave .. +31 (4 loads);
    // lane l covers row base + l/8, slot l%8
    const bool aload = 16 * wave < rows;
    const int slot = lane & 7, rsub = lane >> 3;
    const float* asrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 16 * wave + 8 * i + rsub;
        asrc[i] = x + (int64_t)s_src[r] * K + 4 * (slot ^ (r & 7));
    }
    // (the weights from a uniform base; a lane's part is the same in each load)
    const float* wbase = packed + (3 * (int64_t)e + (GATEUP ? wave >> 1 : 2)) * hidden * inter +
                         (n0 + (GATEUP ? 32 * (wave & 1) : 32 * wave)) * K;
    const uint32_t woff = 4u * (uint32_t)(rsub * K + 4 * (slot ^ rsub));
    const int nk = K / kFBK;
    auto issue = [&](int sl, int ks) {
        char* st = ring[sl];
        const int64_t k0 = (int64_t)ks * kFBK;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            dma16_off(wbase + 8 * i * (int64_t)K + k0, woff, st + kFBM * kFRow + (32 * wave + 8 * i) * kFRow);
        if (aload)
#pragma unroll
            for (int i = 0; i < 2; ++i) dma16(asrc[i] + k0, st + (16 * wave + 8 * i) * kFRow);
    };
    // the sums of the first parts' products, and of the seven others' (2^-7 of
    // them: their roundings do not count), apart
    f4 acc[kFRF][2], low[kFRF][2];
    const int g = lane >> 4, li = lane & 15;
    // this lane's weight rows of the stage: (gate/up) 16*wave + li and
    // 64 + 16*wave + li, (down) 32*wave + li, +16; all of them li mod 8
    const int b0 = GATEUP ? 16 * wave + li : 32 * wave + li;
    const int b1 = b0 + (GATEUP ? 64 : 16);
    const int c0 = 16 * ((2 * g) ^ (li & 7)), c1 = 16 * ((2 * g + 1) ^ (li & 7));
#pragma unroll
    for (int r = 0; r < kFRF; ++r) acc[r][0] = acc[r][1] = low[r][0] = low[r][1] = f4{};
    // stage ks: landed for every wave, and stage ks-1 fully read
    auto stage = [&](int ks) __attribute__((always_inline)) {
        wait_vmcnt<0>();
        lds_barrier();
        if (ks + 1 < nk) issue((ks + 1) % kFSlots, ks + 1);
        return (const char*)ring[ks % kFSlots];
    };
    issue(0, 0);
    for (int ks = 0; ks < nk; ++ks) {
        const char* st = stage(ks);
        const char* wst = st + kFBM * kFRow;
        bf8 wp[2][3];
        split_bf16(*reinterpret_cast<const f4*>(wst + b0 * kFRow + c0),
                   *reinterpret_cast<const f4*>(wst + b0 * kFRow + c1), wp[0]);
        split_bf16(*reinterpret_cast<const f4*>(wst + b1 * kFRow + c0),
                   *reinterpret_cast<const f4*>(wst + b1 * kFRow + c1), wp[1]);
#pragma unroll
        for (int r = 0; r < kFRF; ++r) {
            if (16 * r >= rows) break;  // (uniform)
            const char* ast = st + (16 * r + li) * kFRow;
            bf8 xp[3];
            split_bf16(*reinterpret_cast<const f4*>(ast + c0), *reinterpret_cast<const f4*>(ast + c1), xp);
            // the parts' products, the smallest first
#pragma unroll
            for (int sum = 3; sum >= 1; --sum)
#pragma unroll
                for (int i = min(sum, 2); i >= max(0, sum - 2); --i)
#pragma unroll
                    for (int f = 0; f < 2; ++f)
                        low[r][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xp[i], wp[f][sum - i], low[r][f], 0, 0, 0);
#pragma unroll
            for (int f = 0; f < 2; ++f)
                acc[r][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xp[0], wp[f][0], acc[r][f], 0, 0, 0);
        }
    }
    bool bad = false;
#pragma unroll
    for (int r = 0; r < kFRF; ++r) {
        if (16 * r >= rows) break;
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                acc[r][f][v] = kFUnscale * __fadd_rn(acc[r][f][v], low[r][f][v]);
                low[r][f][v] = 0.0f;
                bad = bad || !(fabsf(acc[r][f][v]) < __builtin_inff());
            }
    }
    if (bad) s_bad = 1;
    __syncthreads();  // (every stage fully read, too)
    if (s_bad) {
        // lane (g, i) holds k = 8 g + 4 q + j in step (q, j)
        issue(0, 0);
        for (int ks = 0; ks < nk; ++ks) {
            const char* st = stage(ks);
            const char* wst = st + kFBM * kFRow;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int c = q ? c1 : c0;
                const f4 w0 = *reinterpret_cast<const f4*>(wst + b0 * kFRow + c);
                const f4 w1 = *reinterpret_cast<const f4*>(wst + b1 * kFRow + c);
#pragma unroll
                for (int r = 0; r < kFRF; ++r) {
                    if (16 * r >= rows) break;  // (uniform)
                    const f4 xv = *reinterpret_cast<const f4*>(st + (16 * r + li) * kFRow + c);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        low[r][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j], w0[j], low[r][0], 0, 0, 0);
                        low[r][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j], w1[j], low[r][1], 0, 0, 0);
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < kFRF; ++r)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    acc[r][f][v] = fabsf(acc[r][f][v]) < __builtin_inff() ? acc[r][f][v] : low[r][f][v];
    }
    // D of a fragment: lane (g, i) holds rows 4 g .. 4 g + 3 of column i
#pragma unroll
    for (int rf = 0; rf < kFRF; ++rf) {
        if (16 * rf >= rows) break;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * rf + 4 * g + v;
            if (r >= rows) continue;
            float* orow = out + (g0 + r) * (int64_t)N + n0;
            if (GATEUP) {
                orow[16 * wave + li] = __fmul_rn(hm_silu(acc[rf][0][v]), acc[rf][1][v]);
            } else {
                orow[32 * wave + li] = acc[rf][0][v];
                orow[32 * wave + 16 + li] = acc[rf][1][v];
            }
        }
    }
}

}  // namespace

// Shapes the FP32 MFMA kernels take (16-byte aligned operands; eight rows of K
// floats within a 32-bit offset).
bool hm_f32_mfma_gateup_ok(int64_t H, int64_t I) {
    return H % kFBK == 0 && I % (kFBN / 2) == 0 && H <= (1 << 26) && I <= INT_MAX / 4;
}
bool hm_f32_mfma_down_ok(int64_t H, int64_t I) {
    return I % kFBK == 0 && H % kFBN == 0 && H <= INT_MAX / 4 && I <= (1 << 26);
}

int hm_launch_gateup_f32_mfma(const hm_layer* L, const float* hidden, const int32_t* counts,
                              const int32_t* offsets, const int32_t* perm_tokens, int64_t R,
                              int64_t max_tiles, float* z, hipStream_t stream) {
    const int64_t nbn = L->intermediate / (kFBN / 2);
    if (R > INT_MAX || max_tiles > ((1 << 24) - 8) / nbn) return HM_ERR_OVERFLOW;  // 2^32 threads
    const dim3 grid((unsigned)((max_tiles * nbn + 7) / 8 * 8));
    HM_STAGE_LAUNCH(true, true, expert_f32_mfma_kernel<true>, grid, dim3(kFThreads), 0, stream,
                    hidden, (int)L->hidden, (int)L->intermediate, (int)L->experts,
                    static_cast<const float*>(L->packed), (int)L->hidden, (int)L->intermediate,
                    counts, offsets, perm_tokens, (int)nbn, z);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_launch_down_f32_mfma(const hm_layer* L, const float* z, const int32_t* counts,
                            const int32_t* offsets, int64_t R, int64_t max_tiles, float* y,
                            hipStream_t stream) {
    const int64_t nbn = L->hidden / kFBN;
    if (R > INT_MAX || max_tiles > ((1 << 24) - 8) / nbn) return HM_ERR_OVERFLOW;  // 2^32 threads
    const dim3 grid((unsigned)((max_tiles * nbn + 7) / 8 * 8));
    hipLaunchKernelGGL(expert_f32_mfma_kernel<false>, grid, dim3(kFThreads), 0, stream, z,
                       (int)L->intermediate, (int)L->hidden, (int)L->experts,
                       static_cast<const float*>(L->packed), (int)L->hidden,
                       (int)L->intermediate, counts, offsets, nullptr, (int)nbn, y);
    HM_LAUNCHED();
    return HM_OK;
}
