// hm_gemm_mfma.hip -- grouped INT8-MFMA expert GEMMs for gfx950.
//
// The activation operand is L fixed-point digit planes with one scale per
// row (hm_device.h); every plane meets the same weight fragment in one
// v_mfma_i32_32x32x32_i8, so each plane's int32 partial over the whole row
// is exact, and the epilogues recombine them (hm_recombine) exactly as the
// generic kernels and the CPU restatement do.  Weights are 1 KB tiles in
// MFMA B-operand order (hm_tile_offset): one 16-byte-per-lane load of a
// contiguous kilobyte is one B fragment.
//
// Operand layout of v_mfma_i32_32x32x32_i8: lane l supplies 16 bytes of row
// l % 32 of A and of column l % 32 of B, K bytes 16 (l / 32) .. +15 of the
// 32-wide step; its 16 int32 results are column l % 32, rows
// 8 (v / 4) + 4 (l / 32) + v % 4 (v = 0..15).
//
// Persistent kernels, one workgroup per CU:
//   ring_gemm_kernel<L, false> (gate/up): 8 wave64s (two per SIMD), A (the
//            token rows' X digit planes, gathered by perm_tokens) and B both
//            staged through an LDS ring by DMA; epilogue g and u -> floats
//            (the SwiGLU runs in the Z quantisation pass, hm_gemm.hip).
//   ring_gemm_kernel<L, true> (down): the same kernel on the grouped rows'
//            Z digit planes and the down tiles; epilogue y -> floats.
//   ring_gemm_ragged_kernel: both for shapes off the tile grid.
//
// Tile order: tiles are numbered m-tile major, column block minor, and split
// into 8 contiguous ranges, one per XCD (workgroup i runs on XCD i % 8), so the
// column blocks of an m-tile (sharing A rows) and the m-tiles of one expert
// (sharing B tiles) meet in one XCD's L2.  In an expert's partial last tile, the
// waves whose rows all lie past its last row skip their MFMAs.
#include "hm_device.h"
#include "hm_lds_dma.h"

#include <limits.h>

#include <type_traits>

namespace {

constexpr int kXcds = 8;
constexpr int kMaxExperts = 256;    // expert tables live in LDS

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

template <int N>
__device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N <= 63, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ v16i mfma32(v4i a, v4i b, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// Exclusive prefix of the m-tiles of every expert (ceil(count / bm)) into
// prefix[0..E], prefix[E] = total.  One full wave.
// Experts with at most `skinny` rows get no tiles (skinny_split_kernel
// takes them).
__device__ __forceinline__ void tile_prefix(const int32_t* cnt, int E, int bm, int skinny,
                                            int32_t* prefix) {
    const int lane = threadIdx.x & (HM_WAVE - 1);
    int base = 0;
    for (int c0 = 0; c0 < E; c0 += HM_WAVE) {
        const int e = c0 + lane;
        const int n = e < E && cnt[e] > skinny ? (cnt[e] + bm - 1) / bm : 0;
        int incl = n;
#pragma unroll
        for (int sft = 1; sft < HM_WAVE; sft <<= 1) {
            const int o = __shfl_up(incl, sft, HM_WAVE);
            if (lane >= sft) incl += o;
        }
        if (e < E) prefix[e] = base + incl - n;
        base += __shfl(incl, HM_WAVE - 1, HM_WAVE);
    }
    if (lane == 0) prefix[E] = base;
}

// Expert owning global m-tile gm: the last expert whose first tile is <= gm
// (experts with no tiles share their successor's start and are skipped).
// Every lane of the wave must be active.
__device__ __forceinline__ int locate_expert(const int32_t* prefix, int E, int gm) {
    const int lane = threadIdx.x & (HM_WAVE - 1);
    int n = 0;
    for (int c0 = 0; c0 < E; c0 += HM_WAVE) {
        const int e = c0 + lane;
        n += __popcll(__ballot(e < E && prefix[e] <= gm));
    }
    return __builtin_amdgcn_readfirstlane(n - 1);
}

// The workgroup's tiles: jbeg, jbeg + step, ... < jend of its XCD's range.
struct TileRange {
    int jbeg, jend, step, ntiles;
};
__device__ __forceinline__ TileRange tile_range(int total) {
    TileRange t;
    const int per = (total + kXcds - 1) / kXcds;
    const int x = blockIdx.x % kXcds;
    t.step = gridDim.x / kXcds;
    t.jbeg = x * per + blockIdx.x / kXcds;
    t.jend = min((x + 1) * per, total);
    t.ntiles = t.jbeg < t.jend ? (t.jend - t.jbeg + t.step - 1) / t.step : 0;
    return t;
}

struct TileInfo {
    int e, nrows, g0, n0;
};

// ===========================================================================
// Skinny groups: bounded split-K.  An expert with at most kSkinnyRows = 32
// grouped rows (a cold expert; most experts of a mid-size batch) would
// fill a tile of BM rows mostly with padding, and the tile still streams
// every row of its A stages.  Such experts skip the tile kernels
// (tile_prefix) and come here: one workgroup per (expert, kSkCB column
// blocks of 32); its A rows (all K, the L digit planes) go to LDS once, in
// MFMA operand order, and its 8 waves are kSkCB column blocks x kSkP K
// parts.  Each wave streams its block's weight tiles over its K part and
// runs v_mfma_i32_32x32x32_i8 on its own accumulators; the parts' int32
// limb partials meet in LDS in part order (integer addition: exact, so the
// partials, and hence the epilogue's floats, equal the tile kernels' bit
// for bit).  K is split into a bounded number of parts as the reference's
// split-K does (P = min(8, ceil(K/512)), Int8GemmPlan.cpp:29-53, reduced in
// a fixed order, CudaKernels.cu:53-107), here kSkP = 2 within a workgroup.
//   GU    gate and up (NP = 2): A = the X digit planes of the rows' tokens
//         (perm_tokens; hm_dlay_x), out = gu [R x 2I];
//   down  (NP = 1): A = the Z digit planes of the grouped rows (hm_dlay_z),
//         out = y.
// LDS: the A rows, L x 32 x K bytes, reused for the partials (skinny_lds).
// ===========================================================================
constexpr int kSkinnyRows = 32;   // one 32-row fragment
constexpr int kSkWaves = 8;
constexpr int kSkThreads = 64 * kSkWaves;
constexpr int kSkP = 2;           // K parts
constexpr int kSkCB = kSkWaves / kSkP;  // column blocks per workgroup
constexpr int kSkLds = 131072;    // A bytes in LDS: L * 32 * K
constexpr int kSkDepth = 4;       // K steps of weights in flight per wave

template <int L, bool GU>
__global__ __launch_bounds__(kSkThreads) void skinny_split_kernel(
    const int8_t* __restrict__ adig, const float* __restrict__ ascale,
    const int32_t* __restrict__ adsum, int arows, const int32_t* __restrict__ perm_tokens,
    int K, int N, int H, int I, const int8_t* __restrict__ packed,
    const float* __restrict__ scale, const int32_t* __restrict__ zp,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
    float* __restrict__ out) {
    constexpr int NP = GU ? 2 : 1;
    extern __shared__ __attribute__((aligned(1024))) int8_t s_a[];   // [L][KT][32 rows][32 B]
    __shared__ int32_t s_arow[32];
    const int e = blockIdx.y;
    const int nrows = counts[e];
    if (nrows == 0 || nrows > kSkinnyRows) return;          // (uniform)
    const int g0 = offsets[e];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KT = K / 32;
    if (tid < 32) {
        const int g = g0 + min(tid, nrows - 1);  // rows past the group repeat its last
        s_arow[tid] = GU ? perm_tokens[g] : g;
    }
    __syncthreads();
    // the A rows into LDS: one wave-wide 16-byte load per (plane, K step):
    // lane -> row lane/2, half lane%2 (32 rows x 32 bytes, MFMA order)
    {
        const int arow = s_arow[lane >> 1];
        const hm_dlay lay = GU ? hm_dlay_x(L, K) : hm_dlay_z(L, arows);
        for (int q = wave; q < L * KT; q += kSkWaves) {
            const int l = q / KT, kt = q - l * KT;
            dma16(adig + hm_dlay_off(lay, l, arow, 32 * kt + 16 * (lane & 1)), s_a + 1024 * q);
        }
    }
    // this wave's column block and K part
    const int cbl = wave % kSkCB, part = wave / kSkCB;
    const int cb = blockIdx.x * kSkCB + cbl;                // output columns 32 cb .. +31
    const int kt0 = part * KT / kSkP, kt1 = (part + 1) * KT / kSkP;
    const bool live = 32 * cb < N;                          // (uniform per wave)
    const int8_t* bsrc[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p)
        bsrc[p] = packed + hm_proj_offset(e, GU ? p : 2, H, I) +
                  (int64_t)min(cb, N / 32 - 1) * KT * 1024 + 16 * lane;
    // weights kSkDepth steps ahead (a step past the part re-reads its last)
    v4i fb[kSkDepth][NP];
#pragma unroll
    for (int d = 0; d < kSkDepth; ++d)
#pragma unroll
        for (int p = 0; p < NP; ++p)
            fb[d][p] = *reinterpret_cast<const v4i*>(bsrc[p] + (int64_t)min(kt0 + d, kt1 - 1) * 1024);
    vm_wait<0>();   // this wave's A loads (the first weights land about as soon)
    lds_barrier();  // every wave's
    v16i acc[L][NP];
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int p = 0; p < NP; ++p) acc[l][p] = v16i{};
    const int aoff = 32 * (lane & 31) + 16 * (lane >> 5);
    for (int kt = kt0; kt < kt1; kt += kSkDepth) {
#pragma unroll
        for (int d = 0; d < kSkDepth; ++d) {
            if (kt + d < kt1) {
                v4i fa[L];
#pragma unroll
                for (int l = 0; l < L; ++l)
                    fa[l] = *reinterpret_cast<const v4i*>(s_a + 1024 * (l * KT + kt + d) + aoff);
#pragma unroll
                for (int l = 0; l < L; ++l)
#pragma unroll
                    for (int p = 0; p < NP; ++p) acc[l][p] = mfma32(fa[l], fb[d][p], acc[l][p]);
            }
#pragma unroll
            for (int p = 0; p < NP; ++p)
                fb[d][p] = *reinterpret_cast<const v4i*>(
                    bsrc[p] + (int64_t)min(kt + d + kSkDepth, kt1 - 1) * 1024);
        }
    }
    // the parts' partials meet in LDS (the A copy is no longer read)
    __syncthreads();
    int32_t* s_p = reinterpret_cast<int32_t*>(s_a);          // [part-1][cbl][L][NP][16][64]
    constexpr int PW = L * NP * 16 * HM_WAVE;                // ints per wave
    if (part > 0) {
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    s_p[((part - 1) * kSkCB + cbl) * PW + ((l * NP + p) * 16 + v) * HM_WAVE + lane] = acc[l][p][v];
    }
    __syncthreads();
    if (part > 0 || !live) return;
#pragma unroll
    for (int q = 1; q < kSkP; ++q)
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    acc[l][p][v] += s_p[((q - 1) * kSkCB + cbl) * PW + ((l * NP + p) * 16 + v) * HM_WAVE + lane];
    // epilogue, as the tile kernels': result register v of lane m is row
    // 8 (v/4) + 4 (m/32) + v%4, column m%32
    const int zpa = zp[3 * e + (GU ? 0 : 2)], zpb = GU ? zp[3 * e + 1] : 0;
    const float sa = scale[3 * e + (GU ? 0 : 2)], sb = GU ? scale[3 * e + 1] : 0.0f;
    const int64_t n = 32 * (int64_t)cb + (lane & 31);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row >= nrows) continue;
        const int arow = s_arow[row];
        const float asc = ascale[arow];
        int pa[L], pb[L];
#pragma unroll
        for (int l = 0; l < L; ++l) {
            pa[l] = acc[l][0][v];
            pb[l] = acc[l][NP - 1][v];
        }
        if (zpa != 0 || zpb != 0) {
#pragma unroll
            for (int l = 0; l < L; ++l) {
                const int ds = adsum[(int64_t)l * arows + arow];
                pa[l] -= zpa * ds;
                pb[l] -= zpb * ds;
            }
        }
        if (GU) {
            const float fg = __fmul_rn(asc, sa), fu = __fmul_rn(asc, sb);
            float* grow = out + (int64_t)(g0 + row) * (2 * (int64_t)I) + n;
            grow[0] = __fmul_rn(hm_recombine(pa, L), fg);
            grow[I] = __fmul_rn(hm_recombine(pb, L), fu);
        } else {
            out[(int64_t)(g0 + row) * N + n] = __fmul_rn(hm_recombine(pa, L), __fmul_rn(asc, sa));
        }
    }
}

// Dynamic LDS of the skinny kernel: the A rows, or the K parts' partials
// (parts 1 .. kSkP-1, 16 ints per lane per accumulator) if larger.
size_t skinny_lds(int64_t K, int32_t limbs, bool gu) {
    const size_t a = (size_t)limbs * 32 * K;
    const size_t p = (size_t)(kSkP - 1) * kSkCB * limbs * (gu ? 2 : 1) * 16 * HM_WAVE * sizeof(int32_t);
    return a > p ? a : p;
}

// Whether the skinny kernel takes this projection: its LDS fits and K
// splits into whole K steps.
bool skinny_ok(int64_t K, int64_t N, int32_t limbs, bool gu) {
    return skinny_lds(K, limbs, gu) <= (size_t)kSkLds && K % 32 == 0 && K / 32 >= kSkP &&
           N % 32 == 0;
}

template <int L, bool GU>
int launch_skinny(const hm_layer* layer, const int8_t* adig, const float* ascale,
                  const int32_t* adsum, int64_t arows, const int32_t* perm_tokens,
                  const int32_t* counts, const int32_t* offsets, float* out, hipStream_t stream,
                  bool timed_first) {
    const int64_t H = layer->hidden, I = layer->intermediate;
    const int64_t K = GU ? H : I, N = GU ? I : H;
    const dim3 grid((unsigned)((N / 32 + kSkCB - 1) / kSkCB), (unsigned)layer->experts);
    const size_t lds = skinny_lds(K, L, GU);
    HM_STAGE_LAUNCH(timed_first, false, (skinny_split_kernel<L, GU>), grid, dim3(kSkThreads), lds,
                    stream, adig, ascale, adsum, (int)arows, perm_tokens, (int)K, (int)N, (int)H,
                    (int)I, static_cast<const int8_t*>(layer->packed), layer->scale,
                    layer->zero_point, counts, offsets, out);
    HM_LAUNCHED();
    return HM_OK;
}

int persistent_grid() {
    static int cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    if (cached[dev] == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        cached[dev] = cus;
    }
    const int g = cached[dev] / kXcds * kXcds;
    return g < kXcds ? kXcds : g;
}

// ===========================================================================
// gate/up: a ring kernel of its own.  8 wave64s per workgroup (two per
// SIMD, 256 registers each), both operands staged through LDS by DMA, so
// while one wave of a SIMD waits (for a stage, or in its epilogue) the other
// keeps the matrix pipe busy.  Tile = BM grouped rows x (128 gate + 128 up)
// weight columns; wave (wr, wc) owns rows [32 WR wr, +32 WR) and gate and up
// columns [32 WCP wc, +32 WCP).  Per ring stage of 64 K bytes:
//   A  the L digit planes of the tile rows (gathered by perm_tokens), in
//      fragments of 32 rows x 64 bytes, two wave-wide 16-byte DMAs each
//      (lane: row 16 h + lane/4, chunk (lane%4) ^ ((lane/16)%4)), read back
//      bank-conflict free with the swizzle of gu_frag_read_offset; at two
//      planes (gate/up) each DMA instead moves 8 rows' whole 128-byte lines
//      (both planes of the stage, adjacent in the X layout) and the reads
//      follow gu_pair_read_offset;
//   B  the 8 weight fragments (4 gate, 4 up column blocks of 32), each the
//      two 1 KB operand-order tiles (hm_tile_offset) of the stage's K steps,
//      one contiguous DMA each and read back at 16 lane.
// The stage's loads are spread over the waves, LPW per wave (the last
// round only on the waves it reaches); a step refills the slot read two
// steps earlier, so its barrier leaves the previous step's fragment reads
// in flight (the K loop below).
// Epilogue: the dequantised g and u values (z = silu(g) * u and the Z digits
// follow in one pass over the rows at full occupancy, hm_gemm.hip).
// ===========================================================================
constexpr int kGuWaves = 8;
constexpr int kGuThreads = 64 * kGuWaves;
constexpr int kGuKB = 64;                   // K bytes per ring stage: two MFMA K steps
constexpr int kGuStages = 4;                // ring stages
constexpr int kGuFrag = 32 * kGuKB;         // bytes of one fragment of a stage
constexpr int kGuN = 128;                   // columns per projection per tile

__device__ __forceinline__ int gu_frag_load_row(int lane, int hf) { return 16 * hf + (lane >> 2); }
__device__ __forceinline__ int gu_frag_load_chunk(int lane) { return (lane & 3) ^ ((lane >> 4) & 3); }
// A fragment reader of K step h: lane m (row r = m%32, chunk c = 2h + m/32)
// at 1024 (r/16) + 16 (4 (r%16) + (c ^ ((r/4)%4))); over any 16 consecutive
// lanes these are 16 distinct 16-byte bank groups.
__device__ __forceinline__ int gu_frag_read_offset(int lane, int h) {
    const int r = lane & 31, c = 2 * h + (lane >> 5);
    return 1024 * (r >> 4) + 16 * (4 * (r & 15) + (c ^ ((r >> 2) & 3)));
}
// The paired (L = 2, gate/up) fragment reader: plane l, K step h, lane m
// (row r = m%32, 16-byte piece c = 4 l + 2 h + m/32 of the row's 128 bytes)
// at 128 r + 16 (c ^ ((r/2)%8)) in the 32-row block; over any 16
// consecutive lanes these are 16 distinct 16-byte bank groups.
__device__ __forceinline__ int gu_pair_read_offset(int lane, int h, int l) {
    const int r = lane & 31, c = 4 * l + 2 * h + (lane >> 5);
    return 128 * r + 16 * (c ^ ((r >> 1) & 7));
}
__device__ __forceinline__ v4i lds16(const int8_t* p) { return *reinterpret_cast<const v4i*>(p); }

template <int L>
struct GateUpTile {
    static constexpr int WR = 1;                        // 32-row fragments per wave
    static constexpr int WCP = L >= 3 ? 1 : 2;          // gate (and up) fragments per wave
    static constexpr int NWC = kGuN / 32 / WCP;         // waves across the columns
    static constexpr int NWR = kGuWaves / NWC;          // waves across the rows
    static constexpr int BM = 32 * WR * NWR;            // 128 rows (64 at three limbs)
    static constexpr int NA = L * BM / 32;              // A fragments per stage
    static constexpr int NB = 2 * kGuN / 32;            // 8 B fragments (4 gate, 4 up)
    static constexpr int NF = NA + NB;
    static constexpr int NL = 2 * NF;                   // wave-wide loads per stage
    static constexpr int LPW = (NL + kGuWaves - 1) / kGuWaves;
    static constexpr int STAGE = NF * kGuFrag;
};

// DN = false: gate/up, A = X digit planes (hm_dlay_x: [T][H/64][L][64])
// gathered by perm_tokens, out = gu [R x 2I] (tile: 128 gate + 128 up
// columns).  At L = 2 the A load units are whole 128-byte lines (a row's two
// planes of the stage), 8 rows a unit, stored at row r's 128 bytes with the
// 16-byte pieces rotated by (r / 2) % 8 (the paired fragment order, read
// conflict-free at gu_pair_read_offset); otherwise 16 rows of one plane's
// 64 bytes a unit (gu_frag_load_row/chunk).
// DN = true: down, A = Z digit planes (hm_dlay_z: [I/64][L][R][64]) of the
// grouped rows themselves (a 16-row load unit is one contiguous kilobyte),
// out = y [R x H] (tile: 256 down columns; the "gate" half of the gate/up
// tile is its first 128 columns, the "up" half the next).
// RAG = true: shapes off the tile grid, with the same integers and floats.
// K is walked in whole 64-byte chunks: the digits past K are zeros (the
// quantisers write them), and where the weights' last 32-wide tile is the
// first half of a stage, its second half re-reads that tile (against zero
// digits).  Column blocks past the last re-read it, and columns past N are
// not stored.  A form of its own so that the aligned shapes keep their loop
// and registers.  The generic kernels (one lane per output, byte loads) took
// such shapes before: 201 tokens, 60 experts top-4, H = 1024, I = 704: the
// whole block 2778 -> 150 us, 71 with today's router (gate/up 28, down 14).
template <int L, bool DN, bool RAG>
__device__ __forceinline__ void ring_gemm_body(
    const int8_t* __restrict__ xdig, const float* __restrict__ xscale,
    const int32_t* __restrict__ xdsum, int tokens, int H, int I, int experts,
    const int8_t* __restrict__ packed, const float* __restrict__ scale,
    const int32_t* __restrict__ zp, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ perm_tokens, int skinny,
    float* __restrict__ gu) {
    using T = GateUpTile<L>;
    // inner and output dimensions of the projection(s), output columns per
    // tile, the out row stride and the offset of the tile's second half
    const int K = RAG ? (int)hm_pad64(DN ? I : H) : (DN ? I : H), N = DN ? H : I;
    constexpr int TN = DN ? 2 * kGuN : kGuN;
    const int64_t ldo = DN ? (int64_t)N : 2 * (int64_t)N;
    const int half = DN ? kGuN : N;
    constexpr int PG = DN ? 2 : 0, PU = DN ? 2 : 1;  // the halves' projections
    constexpr int BM = T::BM, NA = T::NA, NL = T::NL, LPW = T::LPW, WR = T::WR, WCP = T::WCP,
                  NWC = T::NWC, STAGE = T::STAGE;
    constexpr int RW = BM / HM_WAVE;  // waves that move one value per tile row
    constexpr int kS = kGuStages;
    __shared__ __attribute__((aligned(1024))) int8_t ring[kS * STAGE];
    __shared__ int32_t s_prefix[kMaxExperts + 1];
    __shared__ int32_t s_off[kMaxExperts], s_cnt[kMaxExperts];
    __shared__ float s_sg[kMaxExperts], s_su[kMaxExperts];
    __shared__ int32_t s_zg[kMaxExperts], s_zu[kMaxExperts];
    __shared__ __attribute__((aligned(16))) int32_t s_rt[2][BM];     // token of each tile row
    __shared__ __attribute__((aligned(16))) float s_xs[2][BM];       // its activation scale
    __shared__ __attribute__((aligned(16))) int32_t s_xd[2][L][BM];  // its digit sums

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / NWC, wc = wave % NWC;
    const int E = experts;
    for (int e = tid; e < E; e += kGuThreads) {
        s_cnt[e] = counts[e];
        s_off[e] = offsets[e];
        s_sg[e] = scale[3 * e + PG];
        s_su[e] = scale[3 * e + PU];
        s_zg[e] = zp[3 * e + PG];
        s_zu[e] = zp[3 * e + PU];
    }
    __syncthreads();
    if (wave == 0) tile_prefix(s_cnt, E, BM, skinny, s_prefix);
    __syncthreads();
    const int nbn = RAG ? (N + TN - 1) / TN : N / TN;
    const TileRange tr = tile_range(s_prefix[E] * nbn);
    if (tr.ntiles == 0) return;
    const int nk = K / kGuKB;
    const int64_t tiles_k = hm_pad32(DN ? I : H) / 32;  // K tiles of one 32-column block
    const int last_cb = (int)(hm_pad32(N) / 32) - 1;    // (RAG)
    // (RAG) the stage whose second K half has no tile of its own
    const int odd_ks = (tiles_k & 1) ? nk - 1 : -1;

    auto info = [&](int i) __attribute__((always_inline)) {
        const int j = tr.jbeg + i * tr.step;
        const int gm = j / nbn;
        TileInfo t;
        t.e = locate_expert(s_prefix, E, gm);
        const int mt = gm - s_prefix[t.e];
        t.g0 = s_off[t.e] + mt * BM;
        t.nrows = min(BM, s_cnt[t.e] - mt * BM);
        t.n0 = (j % nbn) * TN;
        return t;
    };
    // A rows of the tile rows: their tokens (gate/up) or the grouped rows
    // themselves (down); rows past nrows repeat the last row
    auto fetch_rows = [&](const TileInfo& t, int m) __attribute__((always_inline)) {
        if (wave < RW) {
            const int r = HM_WAVE * wave + lane;
            if constexpr (DN) s_rt[m][r] = t.g0 + min(r, t.nrows - 1);
            else dma4(perm_tokens + t.g0 + min(r, t.nrows - 1), &s_rt[m][HM_WAVE * wave]);
        }
    };
    // activation scales and digit sums of those tokens (needs s_rt[m])
    auto fetch_row_meta = [&](int m) __attribute__((always_inline)) {
        if (wave < RW) {
            const int tok = s_rt[m][HM_WAVE * wave + lane];
            dma4(xscale + tok, &s_xs[m][HM_WAVE * wave]);
#pragma unroll
            for (int l = 0; l < L; ++l) dma4(xdsum + (int64_t)l * tokens + tok, &s_xd[m][l][HM_WAVE * wave]);
        }
    };
    // this wave's load units: unit u = fragment u/2, half (K step) u%2.
    // Unit c of wave w is u = w + 8c; when the stage's NL units do not fill
    // every wave's LPW slots, the waves below NFULL issue LPW loads per stage
    // and the others LPW-1.
    constexpr int NFULL = NL - kGuWaves * (LPW - 1);
    static_assert(NFULL >= 1 && NFULL <= kGuWaves, "load units");
    const bool full = wave < NFULL;
    int dst[LPW];
#pragma unroll
    for (int c = 0; c < LPW; ++c) {
        const int u = (wave + kGuWaves * c) % NL;
        dst[c] = (u >> 1) * kGuFrag + 1024 * (u & 1);
    }
    // per-lane sources at stage 0 and their advance per stage (A: the next
    // 64-byte chunk of the digit layout; B: two 1 KB tiles)
    constexpr bool PAIRED = !DN && L == 2;
    const int astep = DN ? L * tokens * kGuKB : L * kGuKB;
    int sstep[LPW];
#pragma unroll
    for (int c = 0; c < LPW; ++c) sstep[c] = ((wave + kGuWaves * c) % NL) / 2 < NA ? astep : 2048;
    auto make_src = [&](const TileInfo& t, int m, const int8_t* (&src)[LPW]) {
        const int ch = gu_frag_load_chunk(lane);
#pragma unroll
        for (int c = 0; c < LPW; ++c) {
            const int u = (wave + kGuWaves * c) % NL;
            const int f = u >> 1, h = u & 1;
            if (f < NA) {
                if constexpr (PAIRED) {
                    // unit u: rows 8 (u % 4) .. +7 of 32-row block u / 4
                    const int r = 8 * (u & 3) + (lane >> 3);
                    const int tok = s_rt[m][32 * (u >> 2) + r];
                    src[c] = xdig + (int64_t)tok * (L * K) + 16 * ((lane & 7) ^ ((r >> 1) & 7));
                } else {
                    const int l = f / (BM / 32), i = f % (BM / 32);
                    const int tok = s_rt[m][32 * i + gu_frag_load_row(lane, h)];
                    src[c] = DN ? xdig + ((int64_t)l * tokens + tok) * kGuKB + 16 * ch
                                : xdig + (int64_t)tok * (L * K) + l * kGuKB + 16 * ch;
                }
            } else {
                const int fb = f - NA;
                int cb = t.n0 / 32 + (DN ? fb : (fb & 3));
                if constexpr (RAG) cb = min(cb, last_cb);
                src[c] = packed + hm_proj_offset(t.e, DN ? 2 : fb >> 2, H, I) +
                         ((int64_t)cb * tiles_k + h) * 1024 + 16 * lane;
            }
        }
    };
    // load c of a stage exists on this wave
    auto has_unit = [&](int c) __attribute__((always_inline)) { return c < LPW - 1 || full; };
    // where load c of stage ks starts
    auto stage_src = [&](const int8_t* const (&src)[LPW], int c, int ks) __attribute__((always_inline)) {
        int64_t o = (int64_t)ks * sstep[c];
        if constexpr (RAG) {
            const int u = (wave + kGuWaves * c) % NL;
            if (ks == odd_ks && (u >> 1) >= NA && (u & 1)) o -= 1024;
        }
        return src[c] + o;
    };
    auto issue = [&](int slot, const int8_t* const (&src)[LPW], int ks) {
        int8_t* st = ring + slot * STAGE;
#pragma unroll
        for (int c = 0; c < LPW; ++c)
            if (has_unit(c)) dma16(stage_src(src, c, ks), st + dst[c]);
    };
    // wait until at most n stages of this wave's loads are in flight
    auto vm_wait_stages = [&](auto nst) __attribute__((always_inline)) {
        constexpr int n = decltype(nst)::value;
        if (full) vm_wait<n * LPW>();
        else vm_wait<n * (LPW - 1)>();
    };

    int rd[2], rdp[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        rd[h] = gu_frag_read_offset(lane, h);
#pragma unroll
        for (int l = 0; l < 2; ++l) rdp[h][l] = gu_pair_read_offset(lane, h, l);
    }
    v4i fa[2][WR][L], fb[2][2 * WCP];
    v16i acc[WR][L][2 * WCP];
    const int8_t* src[LPW];  // per-lane sources of this wave's loads

    // ---- the K loop.  Stream stage s (the tiles' stages back to back) lives
    // in ring slot s % kS.  Step s: wait until this wave's loads of stage s+1
    // have landed, workgroup barrier, refill the slot of stage s-1 with stage
    // s+kS-1, then the MFMAs of stage s (fragments in registers) while the
    // fragments of stage s+1 are read: register set h as soon as the last
    // MFMA of K step h that uses it has issued.  The slot refilled at step s
    // was read during step s-2, so the barrier needs only this wave's older
    // LDS reads complete: the reads of step s-1 stay in flight across it
    // (a barrier that drained them left all eight waves waiting on the
    // LDS together once per stage, the matrix pipes idle).
    constexpr int NJ = 2 * WCP;                 // B fragments per K step
    constexpr int NM = WR * L * NJ;             // MFMAs per K step
    constexpr int RPS = 2 * (WR * L + NJ);      // LDS fragment reads per step
    static_assert(RPS <= 15, "lgkmcnt range");
    auto read_a = [&](int slot, int h, int ii, int l) __attribute__((always_inline)) {
        if constexpr (PAIRED)
            fa[h][ii][l] = lds16(ring + slot * STAGE + (wr * WR + ii) * 2 * kGuFrag + rdp[h][l]);
        else
            fa[h][ii][l] = lds16(ring + slot * STAGE + (l * (BM / 32) + wr * WR + ii) * kGuFrag + rd[h]);
    };
    auto read_b = [&](int slot, int h, int j) __attribute__((always_inline)) {
        const int fbi = j < WCP ? wc * WCP + j : kGuN / 32 + wc * WCP + (j - WCP);
        fb[h][j] = lds16(ring + slot * STAGE + (NA + fbi) * kGuFrag + 1024 * h + 16 * lane);
    };
    // K step h of the current stage; rslot: slot of the stage whose set-h
    // fragments are read meanwhile (-1: none); (h = 0) the step's refill
    // loads into dslot from source stage dks go out after the first MFMAs.
    // The sched_barriers keep this order.
    auto kstep_h = [&](auto hc, auto first, int rslot, int dslot, int dks) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
#pragma unroll
        for (int mi = 0; mi < NM; ++mi) {
            const int ii = mi / (L * NJ), l = (mi / NJ) % L, j = mi % NJ;
            if constexpr (decltype(first)::value)
                acc[ii][l][j] = mfma32(fa[h][ii][l], fb[h][j], v16i{});
            else
                acc[ii][l][j] = mfma32(fa[h][ii][l], fb[h][j], acc[ii][l][j]);
            if (h == 0 && mi < LPW && dslot >= 0 && has_unit(mi))
                dma16(stage_src(src, mi, dks), ring + dslot * STAGE + dst[mi]);
            if (rslot >= 0) {
                if (j == NJ - 1) read_a(rslot, h, ii, l);
                if (ii == WR - 1 && l == L - 1) read_b(rslot, h, j);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (h == 0 && dslot >= 0)
#pragma unroll
            for (int c = NM; c < LPW; ++c)
                if (has_unit(c)) dma16(stage_src(src, c, dks), ring + dslot * STAGE + dst[c]);
    };
    auto read_all = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int ii = 0; ii < WR; ++ii)
#pragma unroll
                for (int l = 0; l < L; ++l) read_a(slot, h, ii, l);
#pragma unroll
            for (int j = 0; j < NJ; ++j) read_b(slot, h, j);
        }
    };

    // ---- stream prologue: tile 0's rows, metadata and first kS-1 stages
    TileInfo cur = info(0);
    int m = 0;
    fetch_rows(cur, 0);
    vm_wait<0>();
    lds_barrier();
    fetch_row_meta(0);
    make_src(cur, 0, src);
    int slot0 = 0;  // ring slot of the current tile's stage 0
#pragma unroll
    for (int s = 0; s < kS - 1; ++s) issue(s, src, s);
    vm_wait_stages(std::integral_constant<int, kS - 2>{});
    lds_barrier();

    for (int i = 0; i < tr.ntiles; ++i) {
        const bool has_next = i + 1 < tr.ntiles;
        const int mn = m ^ 1;
        TileInfo nxt = cur;
        if (has_next) nxt = info(i + 1);
        // a wave whose rows all lie past the tile's last row (an expert's
        // partial last tile) skips its fragment reads and MFMAs
        const bool act = 32 * WR * wr < cur.nrows;
        // Step ks.  Phase A (ks <= nk-kS): refill with this tile's stage
        // ks+kS-1; phase B: with the next tile's stage ks+kS-1-nk.
        auto step = [&](int ks, auto first, auto phase_b, auto active) __attribute__((always_inline)) {
            constexpr bool B = decltype(phase_b)::value, ACT = decltype(active)::value;
            // stage ks+1 of the stream has landed once at most the stages
            // after it that are already issued (ks+2 .. ks+kS-2) are in flight
            if (!B || has_next) vm_wait_stages(std::integral_constant<int, kS - 3>{});
            else if (ks + 1 < nk) vm_wait<0>();
            if constexpr (ACT) lds_barrier_keep<RPS>();
            else lds_barrier();
            const int dslot = !B || has_next ? (slot0 + ks + kS - 1) % kS : -1;
            const int dks = B ? ks + kS - 1 - nk : ks + kS - 1;
            if (decltype(first)::value && has_next) fetch_rows(nxt, mn);
            if constexpr (ACT) {
                const int rslot = ks + 1 < nk ? (slot0 + ks + 1) % kS : -1;
                kstep_h(std::integral_constant<int, 0>{}, first, rslot, dslot, dks);
                kstep_h(std::integral_constant<int, 1>{}, std::false_type{}, rslot, -1, 0);
            } else if (dslot >= 0) {
                issue(dslot, src, dks);
            }
        };
        auto tile_k = [&](auto active) __attribute__((always_inline)) {
            // stage 0's fragments (landed and published by the previous
            // step's barrier)
            if constexpr (decltype(active)::value) read_all(slot0);
            step(0, std::true_type{}, std::false_type{}, active);
            int ks = 1;
#pragma clang loop unroll(disable)
            for (; ks <= nk - kS; ++ks) step(ks, std::false_type{}, std::false_type{}, active);
            if (has_next) {
                // the next tile's loads start now: their sources (its row
                // tokens have landed, a stage issued after them has) and its
                // row metadata
                if (nk < 2 * kS) {
                    vm_wait<0>();
                    lds_barrier();
                }
                make_src(nxt, mn, src);
                fetch_row_meta(mn);
            }
#pragma clang loop unroll(disable)
            for (; ks < nk; ++ks) step(ks, std::false_type{}, std::true_type{}, active);
        };
        if (act) tile_k(std::true_type{});
        else tile_k(std::false_type{});

        // ---- epilogue (the next tile's first kS-2 stages are in flight):
        // g and u into the row's two halves of gu.  The zero-point
        // correction is chosen once per tile (zg, zu are uniform), so no
        // per-element test drags its integer multiplies into the common case.
        auto epilogue = [&](auto with_zp) __attribute__((always_inline)) {
            constexpr bool ZP = decltype(with_zp)::value;
            const int e = cur.e, nrows = cur.nrows;
            const float sg = s_sg[e], su = s_su[e];
            const int zg = s_zg[e], zu = s_zu[e];
            const int col = cur.n0 + 32 * wc * WCP + (lane & 31);  // (RAG) the lane's column
#pragma unroll
            for (int ii = 0; ii < WR; ++ii) {
                const int r0 = 32 * (wr * WR + ii);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int rq = r0 + 8 * q + 4 * (lane >> 5);  // rows rq .. rq+3
                    const float4 sx4 = *reinterpret_cast<const float4*>(&s_xs[m][rq]);
                    int4 ds4[L];
                    if constexpr (ZP) {
#pragma unroll
                        for (int l = 0; l < L; ++l) ds4[l] = *reinterpret_cast<const int4*>(&s_xd[m][l][rq]);
                    }
#pragma unroll
                    for (int t4 = 0; t4 < 4; ++t4) {
                        const int v = 4 * q + t4;
                        const float sx = t4 == 0 ? sx4.x : t4 == 1 ? sx4.y : t4 == 2 ? sx4.z : sx4.w;
                        const float fg = __fmul_rn(sx, sg), fu = __fmul_rn(sx, su);
                        const bool live = rq + t4 < nrows;
                        float* grow = gu + (int64_t)(cur.g0 + rq + t4) * ldo + cur.n0 +
                                      32 * wc * WCP + (lane & 31);
#pragma unroll
                        for (int j = 0; j < WCP; ++j) {
                            int pg[L], pu[L];
#pragma unroll
                            for (int l = 0; l < L; ++l) {
                                pg[l] = acc[ii][l][j][v];
                                pu[l] = acc[ii][l][WCP + j][v];
                            }
                            if constexpr (ZP) {
#pragma unroll
                                for (int l = 0; l < L; ++l) {
                                    const int ds = t4 == 0 ? ds4[l].x : t4 == 1 ? ds4[l].y : t4 == 2 ? ds4[l].z : ds4[l].w;
                                    pg[l] -= zg * ds;
                                    pu[l] -= zu * ds;
                                }
                            }
                            const float g = __fmul_rn(hm_recombine(pg, L), fg);
                            const float u = __fmul_rn(hm_recombine(pu, L), fu);
                            if constexpr (RAG) {
                                if (live && col + 32 * j < N) {
                                    grow[32 * j] = g;
                                    if (!DN || col + kGuN + 32 * j < N) grow[half + 32 * j] = u;
                                }
                            } else if (live) {
                                if constexpr (DN) {
                                    grow[32 * j] = g;
                                    grow[half + 32 * j] = u;
                                } else {
                                    // g | u is read once, by the SwiGLU pass:
                                    // streamed, so that it does not evict the
                                    // operands the other tiles read again
                                    __builtin_nontemporal_store(g, &grow[32 * j]);
                                    __builtin_nontemporal_store(u, &grow[half + 32 * j]);
                                }
                            }
                        }
                    }
                }
            }
        };
        if (act) {
            if ((s_zg[cur.e] | s_zu[cur.e]) != 0) epilogue(std::true_type{});
            else epilogue(std::false_type{});
        }
        // next tile
        slot0 = (slot0 + nk) % kS;
        m = mn;
        cur = nxt;
    }
}

template <int L, bool DN>
__global__ __launch_bounds__(kGuThreads) void ring_gemm_kernel(
    const int8_t* __restrict__ xdig, const float* __restrict__ xscale,
    const int32_t* __restrict__ xdsum, int tokens, int H, int I, int experts,
    const int8_t* __restrict__ packed, const float* __restrict__ scale,
    const int32_t* __restrict__ zp, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ perm_tokens, int skinny,
    float* __restrict__ gu) {
    ring_gemm_body<L, DN, false>(xdig, xscale, xdsum, tokens, H, I, experts, packed, scale, zp, counts, offsets, perm_tokens,
                                    skinny, gu);
}

template <int L, bool DN>
__global__ __launch_bounds__(kGuThreads) void ring_gemm_ragged_kernel(
    const int8_t* __restrict__ xdig, const float* __restrict__ xscale,
    const int32_t* __restrict__ xdsum, int tokens, int H, int I, int experts,
    const int8_t* __restrict__ packed, const float* __restrict__ scale,
    const int32_t* __restrict__ zp, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ perm_tokens, int skinny,
    float* __restrict__ gu) {
    ring_gemm_body<L, DN, true>(xdig, xscale, xdsum, tokens, H, I, experts, packed, scale, zp, counts, offsets, perm_tokens,
                                    skinny, gu);
}

// Shapes of the ring kernel: K in at least kGuStages 64-byte stages.
bool ring_ok(int64_t K, int64_t N, int64_t E, int32_t limbs) {
    // |P_l| <= K * 128 * 255 < 2^31 keeps every limb partial exact: K <= 65536
    return limbs >= 1 && limbs <= 3 && E >= 1 && E <= kMaxExperts && K <= 65536 &&
           N <= (1 << 20) && hm_pad64(K) / kGuKB >= kGuStages;
}
// ... on its tile grid: whole stages and whole column blocks.
bool ring_aligned(int64_t K, int64_t N, int64_t cols) { return K % kGuKB == 0 && N % cols == 0; }

// Down: skinny groups (split K, when asked for), then the tiles of the
// others.
template <int L>
int launch_down(const hm_layer* layer, const int8_t* zdig, const float* zscale,
                const int32_t* zdsum, int64_t R, const int32_t* counts, const int32_t* offsets,
                float* y, bool split_k, hipStream_t stream) {
    if (!ring_ok(layer->intermediate, layer->hidden, layer->experts, L)) return HM_ERR_UNSUPPORTED;
    const bool sk = split_k && skinny_ok(layer->intermediate, layer->hidden, L, false);
    if (sk) {
        const int rc = launch_skinny<L, false>(layer, zdig, zscale, zdsum, R, nullptr, counts,
                                               offsets, y, stream, false);
        if (rc) return rc;
    }
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)persistent_grid()), dim3(kGuThreads), 0, stream,
                           zdig, zscale, zdsum, (int)R, (int)layer->hidden,
                           (int)layer->intermediate, (int)layer->experts,
                           static_cast<const int8_t*>(layer->packed), layer->scale,
                           layer->zero_point, counts, offsets, nullptr, sk ? kSkinnyRows : 0, y);
    };
    if (ring_aligned(layer->intermediate, layer->hidden, 2 * kGuN)) run(ring_gemm_kernel<L, true>);
    else run(ring_gemm_ragged_kernel<L, true>);
    HM_LAUNCHED();
    return HM_OK;
}

template <int L>
int launch_gateup(const hm_layer* layer, const int8_t* xdig, const float* xscale,
                  const int32_t* xdsum, int64_t tokens, const int32_t* counts,
                  const int32_t* offsets, const int32_t* perm_tokens, float* gu, bool split_k,
                  hipStream_t stream) {
    // skinny groups (split K, when asked for; its start opens an armed stage
    // timer), then the tiles of the others
    const bool sk = split_k && skinny_ok(layer->hidden, layer->intermediate, L, true);
    if (sk) {
        const int rc = launch_skinny<L, true>(layer, xdig, xscale, xdsum, tokens, perm_tokens,
                                              counts, offsets, gu, stream, true);
        if (rc) return rc;
    }
    auto run = [&](auto kernel) {
        HM_STAGE_LAUNCH(!sk, false, kernel, dim3((unsigned)persistent_grid()), dim3(kGuThreads), 0,
                        stream, xdig, xscale, xdsum, (int)tokens, (int)layer->hidden,
                        (int)layer->intermediate, (int)layer->experts,
                        static_cast<const int8_t*>(layer->packed), layer->scale,
                        layer->zero_point, counts, offsets, perm_tokens, sk ? kSkinnyRows : 0, gu);
    };
    if (ring_aligned(layer->hidden, layer->intermediate, kGuN)) run(ring_gemm_kernel<L, false>);
    else run(ring_gemm_ragged_kernel<L, false>);
    HM_LAUNCHED();
    return HM_OK;
}

}  // namespace

// Shape preconditions of the MFMA kernels: at least four 64-byte K stages
// (the ring's look-ahead), E <= 256 (tables in LDS), any N.
bool hm_mfma_gateup_ok(int64_t H, int64_t I, int64_t E, int32_t limbs) {
    return ring_ok(H, I, E, limbs);
}

bool hm_mfma_down_ok(int64_t H, int64_t I, int64_t E, int32_t limbs) {
    return ring_ok(I, H, E, limbs);
}

// gu [R x 2I]: the gate and up values of every grouped row (X digits in the
// hm_dlay_x layout).  The first kernel of the gate/up stage (its start opens
// an armed stage timer).
int hm_launch_gateup_i8_mfma(const hm_layer* layer, int32_t limbs, const int8_t* xdig,
                             const float* xscale, const int32_t* xdsum, int64_t tokens,
                             const int32_t* counts, const int32_t* offsets,
                             const int32_t* perm_tokens, int64_t R, float* gu, bool split_k,
                             hipStream_t stream) {
    if (tokens > INT_MAX || R > INT_MAX) return HM_ERR_OVERFLOW;
    switch (limbs) {
    case 1: return launch_gateup<1>(layer, xdig, xscale, xdsum, tokens, counts, offsets, perm_tokens, gu, split_k, stream);
    case 2: return launch_gateup<2>(layer, xdig, xscale, xdsum, tokens, counts, offsets, perm_tokens, gu, split_k, stream);
    case 3: return launch_gateup<3>(layer, xdig, xscale, xdsum, tokens, counts, offsets, perm_tokens, gu, split_k, stream);
    default: return HM_ERR_INVALID;
    }
}

// y [R x H] from the Z digit planes (hm_dlay_z; one scale per row).
int hm_launch_down_i8_mfma(const hm_layer* layer, int32_t limbs, const int32_t* counts,
                           const int32_t* offsets, int64_t R, const int8_t* zdig,
                           const float* zscale, const int32_t* zdsum, float* y, bool split_k,
                           hipStream_t stream) {
    if (R > INT_MAX) return HM_ERR_OVERFLOW;
    switch (limbs) {
    case 1: return launch_down<1>(layer, zdig, zscale, zdsum, R, counts, offsets, y, split_k, stream);
    case 2: return launch_down<2>(layer, zdig, zscale, zdsum, R, counts, offsets, y, split_k, stream);
    case 3: return launch_down<3>(layer, zdig, zscale, zdsum, R, counts, offsets, y, split_k, stream);
    default: return HM_ERR_INVALID;
    }
}
