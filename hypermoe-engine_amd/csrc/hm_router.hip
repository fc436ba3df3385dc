// hm_router.hip -- RMSNorm, router top-k, token permute, gather, combine and
// elementwise kernels for gfx950 (wave64).  Every kernel here reproduces the
// reference CPU arithmetic bit for bit; the comments say how.
#include "hm_device.h"
#include "hm_gemv_slice.h"
#include "hm_lds_dma.h"

#include <limits.h>

#include <type_traits>

namespace {

constexpr int kBlock = 256;
constexpr int kPermChunk = 1024;  // pairs per permutation chunk (kPermThreads)

__device__ __forceinline__ void hm_status_or(int32_t* status, unsigned bits) {
    if (status) atomicOr(reinterpret_cast<unsigned int*>(status), bits);
}

// ---------------------------------------------------------------------------
// A1 RMSNorm (src/transformer/norm/RMSNorm.cpp:65-77), one workgroup per row.
//
// The reference sums double(x)^2 sequentially.  Squares of floats are exact
// in double, so only the summation order differs between a tree sum s_fast
// and the sequential s_seq; both lie within gamma_{n-1} * S of the exact sum
// S (any recursive summation order, Higham eq. 4.4), so
//   s_seq in [s_fast (1 - d), s_fast (1 + d)],  d = 4 gamma_{n-1}/(1-gamma).
// inv(s) = 1/sqrt(s/W + eps) and y(inv) = float(x * inv * g) are monotone
// under IEEE rounding, so an element whose y is equal at both ends of the
// interval equals the reference's y.  If any element of the row is
// ambiguous, the row falls back to the sequential sum (one wave), which is
// the reference computation itself.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double hm_inv_rms(double s, double width, double eps) {
    return 1.0 / sqrt(s / width + eps);
}

// The relative half-width d of the interval around a tree sum of `width`
// squares that holds the sequential sum (above).
__device__ __forceinline__ double hm_rms_sum_slack(int64_t width) {
    const double u = 0x1p-53;
    const double gam = (double)(width - 1) * u / (1.0 - (double)(width - 1) * u);
    return 4.0 * gam / (1.0 - gam);
}

// Sequential FP64 chains.  The references' sums are chains of dependent
// additions s_k = fl(s_{k-1} + p_k), so what a chain costs is the latency of
// such an addition and how its terms reach it.  They come through DPP: the 16
// lanes of a row hold 64 consecutive terms, lane i the terms 4 i .. 4 i + 3, and
// each step is one v_fmac_f64 whose first operand is lane i's term broadcast
// over the row (row_newbcast:i; times 1.0, so the one rounding is the
// addition's), with no LDS round trip, register move or wait between steps.
// Measured, 2000 chains of 64: 5.8 cycles a step (2.4 ns at 2.4 GHz; 2.6 with two
// waves on every CU), where a dependent v_add_f64 takes 8.3 and a v_fma_f64 8.4.
// Each row of 16 lanes runs a chain of its own (four chains a wave; with the
// same terms in every row, every lane gets the sum).  All lanes of the wave
// must be active.  (The leading s_nop covers the DPP read of a register that
// the instruction before the block wrote.)
#define HM_CHAIN4(i)                                                                \
    "v_fmac_f64_dpp %0, %1, %5 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f64_dpp %0, %2, %5 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f64_dpp %0, %3, %5 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f64_dpp %0, %4, %5 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void hm_chain64(double& acc, double p0, double p1, double p2, double p3) {
    asm volatile("s_nop 4\n\t"
                 HM_CHAIN4(0) HM_CHAIN4(1) HM_CHAIN4(2) HM_CHAIN4(3) HM_CHAIN4(4) HM_CHAIN4(5)
                 HM_CHAIN4(6) HM_CHAIN4(7) HM_CHAIN4(8) HM_CHAIN4(9) HM_CHAIN4(10) HM_CHAIN4(11)
                 HM_CHAIN4(12) HM_CHAIN4(13) HM_CHAIN4(14) HM_CHAIN4(15)
                 : "+&v"(acc)
                 : "v"(p0), "v"(p1), "v"(p2), "v"(p3), "v"(1.0));
}
#undef HM_CHAIN4

// The reference's own sum of squares: double(x_k)^2 added in ascending k from
// +0 (terms past the end are +0, which changes no sum of squares).  Every
// lane returns it; xr in LDS or global memory.
__device__ __forceinline__ double hm_rms_sum_seq(const float* xr, int64_t width) {
    const int64_t i = 4 * (threadIdx.x & 15);
    const int64_t last = width - 1;
    auto load = [&](int64_t k0, float (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t k = k0 + i + q;
            v[q] = xr[k < last ? k : last];
            if (k > last) v[q] = 0.0f;
        }
    };
    double s = 0.0;
    float cur[4], nxt[4];
    load(0, cur);
    for (int64_t k0 = 0; k0 < width; k0 += 64) {
        load(k0 + 64, nxt);
        hm_chain64(s, (double)cur[0] * cur[0], (double)cur[1] * cur[1], (double)cur[2] * cur[2],
                   (double)cur[3] * cur[3]);
#pragma unroll
        for (int q = 0; q < 4; ++q) cur[q] = nxt[q];
    }
    return s;
}

__global__ __launch_bounds__(kBlock) void rmsnorm_kernel(
    const float* __restrict__ x, const float* __restrict__ gamma,
    float* __restrict__ y, int64_t width, float eps, int force_seq) {
    extern __shared__ float row_lds[];  // width floats
    __shared__ double red[kBlock / HM_WAVE];
    __shared__ int ambiguous;
    __shared__ double inv_seq;
    const int64_t r = blockIdx.x;
    const float* xr = x + r * width;
    float* yr = y + r * width;
    const int tid = threadIdx.x;
    if (tid == 0) ambiguous = force_seq;
    double local = 0.0;
    for (int64_t i = tid; i < width; i += kBlock) {
        const float v = xr[i];
        row_lds[i] = v;
        local += (double)v * v;
    }
    local = hm_wave_sum_f64(local);
    if ((tid & (HM_WAVE - 1)) == 0) red[tid / HM_WAVE] = local;
    __syncthreads();
    double s_fast = 0.0;
    for (int w = 0; w < kBlock / HM_WAVE; ++w) s_fast += red[w];
    const double d = hm_rms_sum_slack(width);
    const double wd = (double)width, ed = (double)eps;
    const double inv_lo = hm_inv_rms(s_fast * (1.0 + d), wd, ed);
    const double inv_hi = hm_inv_rms(s_fast * (1.0 - d), wd, ed);
    for (int64_t i = tid; i < width; i += kBlock) {
        const float v = row_lds[i];
        const float a = (float)((double)v * inv_lo * (double)gamma[i]);
        const float b = (float)((double)v * inv_hi * (double)gamma[i]);
        if (__float_as_uint(a) == __float_as_uint(b)) {
            yr[i] = a;
        } else {
            ambiguous = 1;
        }
    }
    __syncthreads();
    if (!ambiguous) return;
    if (tid < HM_WAVE) {
        const double s = hm_rms_sum_seq(row_lds, width);
        if (tid == 0) inv_seq = hm_inv_rms(s, wd, ed);
    }
    __syncthreads();
    const double inv = inv_seq;
    for (int64_t i = tid; i < width; i += kBlock) {
        yr[i] = (float)((double)row_lds[i] * inv * (double)gamma[i]);
    }
}

// The same RMSNorm for rows of 256 V floats (16-byte aligned), one wave per
// row and four rows per workgroup: a lane's V 16-byte loads are issued
// together and the row stays in registers (rmsnorm_kernel's strided loop
// waits for each load before the next).  Same bracket, same fallback (a row
// with an ambiguous element, or every row with force_seq, takes the
// sequential sum, its terms read again from the row: about one row in 128 of
// N(0, 1) data, and its chain of W additions sets the kernel's time).
template <int V>
__global__ __launch_bounds__(kBlock) void rmsnorm_wave_kernel(
    const float* __restrict__ x, const float* __restrict__ gamma,
    float* __restrict__ y, int64_t rows, float eps, int force_seq) {
    constexpr int W = 256 * V;
    const int lane = threadIdx.x & (HM_WAVE - 1);
    const int64_t r = (int64_t)blockIdx.x * (kBlock / HM_WAVE) + threadIdx.x / HM_WAVE;
    if (r >= rows) return;
    const float4* xr = reinterpret_cast<const float4*>(x + r * W);
    const float4* g4 = reinterpret_cast<const float4*>(gamma);
    float4* yr = reinterpret_cast<float4*>(y + r * W);
    float4 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = xr[HM_WAVE * j + lane];
    double local = 0.0;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        local += (double)v[j].x * v[j].x;
        local += (double)v[j].y * v[j].y;
        local += (double)v[j].z * v[j].z;
        local += (double)v[j].w * v[j].w;
    }
    const double s_fast = hm_wave_sum_f64(local);  // equal on every lane
    const double d = hm_rms_sum_slack(W);
    const double wd = (double)W, ed = (double)eps;
    const double inv_lo = hm_inv_rms(s_fast * (1.0 + d), wd, ed);
    const double inv_hi = hm_inv_rms(s_fast * (1.0 - d), wd, ed);
    float4 out[V];
    bool amb = false;
    auto one = [&](float xv, float gv, float& o) __attribute__((always_inline)) {
        const float a = (float)((double)xv * inv_lo * (double)gv);
        const float b = (float)((double)xv * inv_hi * (double)gv);
        o = a;
        amb |= __float_as_uint(a) != __float_as_uint(b);
    };
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const float4 g = g4[HM_WAVE * j + lane];
        one(v[j].x, g.x, out[j].x);
        one(v[j].y, g.y, out[j].y);
        one(v[j].z, g.z, out[j].z);
        one(v[j].w, g.w, out[j].w);
    }
    if (force_seq || __ballot(amb) != 0) {
        const float4* xc = xr + (lane & 15);
        double s = 0.0;
        float4 cur = xc[0], nxt = xc[16];
        for (int c = 0; c < W / 64; ++c) {
            const float4 x4 = cur;
            cur = nxt;
            nxt = xc[16 * min(c + 2, W / 64 - 1)];
            hm_chain64(s, (double)x4.x * x4.x, (double)x4.y * x4.y, (double)x4.z * x4.z,
                       (double)x4.w * x4.w);
        }
        const double inv = hm_inv_rms(s, wd, ed);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const float4 g = g4[HM_WAVE * j + lane];
            out[j].x = (float)((double)v[j].x * inv * (double)g.x);
            out[j].y = (float)((double)v[j].y * inv * (double)g.y);
            out[j].z = (float)((double)v[j].z * inv * (double)g.z);
            out[j].w = (float)((double)v[j].w * inv * (double)g.w);
        }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) yr[HM_WAVE * j + lane] = out[j];
}

// ---------------------------------------------------------------------------
// A2 router logits (src/router/CpuRouterBackend.cpp:41-49):
//   logit[t,e] = float(sum_k double(h[t,k]) * double(w[k,e])), k ascending.
// The product of two floats is exact in double, so fma(h, w, acc) rounds
// exactly like the reference's multiply-then-add, and the reference's logit is
// a chain of fused multiply-adds.  The FP64 matrix instructions compute just
// that: for every result, v_mfma_f64_16x16x4_f64 and v_mfma_f64_4x4x4_4b_f64
// add the four products of their k slots to C in ascending order, one fused
// multiply-add each (verified bit for bit against fma chains: 655,360 results
// of 256 steps, narrow, wide and full double operands, no difference; the
// other orders differ in three of four).  So with k slot g of step s holding
// k = 4 s + g, one accumulator from +0 over all of K is the reference's chain:
// no bound, no fallback, nothing kept beside the logits.
//
// What bounds it: FP64 matrix rate for many tokens (4096 x 2048 x 128: 27 us),
// and for few the chain itself: 512 dependent 4 x 4 x 4 steps of 21 cycles (5
// us), the 16 x 16 x 4 form 64 cycles.  One workgroup: 4 waves, 4 C tokens x 64
// experts, a wave 16 experts; C = 1, 2: one, two 4 x 4 x 4 chains (each of its
// four blocks the same four tokens and its own four experts), C = 4, 8: one,
// two 16 x 16 x 4 chains.  W [64 k][64 experts] and h come through a ring of
// stages in LDS by DMA (16-byte where E % 64 == 0 and w is 16-byte aligned,
// else 4-byte), one barrier a stage; row k's 16-float groups are stored
// exchanged by k % 4 and h's rows 68 floats apart, so that the four k slots of
// a lane group read 64 different banks.  C: a workgroup takes 17, 24, 29 and 46
// us at H = 2048 (one a CU; a step's conversions and LDS reads, issued by one
// wave a SIMD, are what lies between these and the chain), so the fewest
// rounds of workgroups times that.
//
// Measured, logits + selection inside a block at H = 2048, E = 128 (before:
// K ranges summed on the matrix cores, an error bound in the select kernel, and
// a second sum and chains for what it left open): 61 tokens 16 + 23 -> 20 + 6
// us, 333 17 + 36 -> 21 + 7 us, 2048 32 + 44 -> 38 + 12 us, 4096 55 + 42 -> 58 +
// 19 us; 201 tokens of H = 1024, E = 60 (one chain per thread before) 87 + 5 ->
// 13 + 4 us.
// ---------------------------------------------------------------------------
constexpr int kCK = 64;   // k per stage
constexpr int kCH = 68;   // floats from one token's h to the next in a stage
typedef double hm_double4 __attribute__((ext_vector_type(4)));

template <int C, bool VEC>
__global__ __launch_bounds__(256) void router_chain_kernel(
    const float* __restrict__ h, const float* __restrict__ w, int64_t tokens, int64_t hidden,
    int experts, float* __restrict__ logits, int32_t* status, int32_t* __restrict__ hist, int hist_n) {
    constexpr int NI = (VEC ? 4 : 16) + C;  // DMA loads per wave and stage
    // ring stages: a stage lasts 340 cycles at C = 1 and 2060 at C = 8, a load
    // from memory about 2000
    constexpr int kCS = !VEC ? 4 : C == 1 ? 8 : C == 2 ? 6 : 4;
    static_assert((kCS - 2) * NI <= 63, "vmcnt");
    constexpr bool BIG = C >= 4;            // 16 x 16 x 4 steps
    constexpr int NT = BIG ? C / 4 : C;     // chains per wave
    __shared__ __attribute__((aligned(1024))) float s_w[kCS][kCK][HM_WAVE];
    __shared__ __attribute__((aligned(1024))) float s_h[kCS][4 * C][kCH];
    // the permutation's chunk histograms, counted by the select kernel
    if (blockIdx.y == 0)
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < hist_n; i += (int64_t)gridDim.x * 256)
            hist[i] = 0;
    const int lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e0 = blockIdx.y * HM_WAVE;
    const int64_t t0 = (int64_t)blockIdx.x * (4 * C);
    const int whole = (int)(hidden / kCK);                  // whole stages
    const int nm = (int)((hidden + kCK - 1) / kCK);
    // The next stage's loads (called in stage order): W rows and C of the
    // tokens' h rows, each from a uniform base, advanced by a stage, and a
    // 32-bit lane offset; in the last, partial stage rows past the end are the
    // last row again (the steps there are masked).
    const int col = VEC ? 4 * (li ^ (4 * g)) : 0;
    const uint32_t wo = VEC ? (uint32_t)(((4 * wave + g) * experts + e0 + col) * 4) : 0;
    const float* wb = w;
    const int64_t wstep = 16 * (int64_t)experts;
    const float* hb[C];
#pragma unroll
    for (int n = 0; n < C; ++n) hb[n] = h + min(t0 + C * wave + n, tokens - 1) * hidden;
    int im = 0, islot = 0;  // the next stage to load and its slot
    auto issue = [&]() __attribute__((always_inline)) {
        uint32_t ho = 4u * (uint32_t)lane;
        if (im < whole) {  // (uniform)
            if constexpr (VEC) {
#pragma unroll
                for (int q = 0; q < 4; ++q) dma16_off(wb + q * wstep, wo, &s_w[islot][16 * q + 4 * wave][0]);
            } else {
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    dma4_off(wb + (16 * wave + q) * (int64_t)experts,
                             4u * (uint32_t)min(e0 + (lane ^ (16 * (q & 3))), experts - 1),
                             &s_w[islot][16 * wave + q][0]);
            }
        } else {
            const int left = (int)(hidden - (int64_t)im * kCK);
            if constexpr (VEC) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    dma16_off(wb, (uint32_t)((min(16 * q + 4 * wave + g, left - 1) * experts + e0 + col) * 4),
                              &s_w[islot][16 * q + 4 * wave][0]);
            } else {
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    dma4_off(wb + min(16 * wave + q, left - 1) * (int64_t)experts,
                             4u * (uint32_t)min(e0 + (lane ^ (16 * (q & 3))), experts - 1),
                             &s_w[islot][16 * wave + q][0]);
            }
            ho = 4u * (uint32_t)min(lane, left - 1);
        }
#pragma unroll
        for (int n = 0; n < C; ++n) {
            dma4_off(hb[n], ho, &s_h[islot][C * wave + n][0]);
            hb[n] += kCK;
        }
        wb += 4 * wstep;
        ++im;
        islot = islot + 1 == kCS ? 0 : islot + 1;
    };
    typedef typename std::conditional<BIG, hm_double4, double>::type Acc;
    Acc acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = Acc{};
    const int woff = HM_WAVE * g + 16 * (wave ^ g) + li;    // W of k slot g, expert 16 wave + li
    const int hoff = kCH * (BIG ? li : lane & 3) + g;       // h of k slot g, the lane's token
    // The operands of four steps (16 k) are a group, group q of a stage in
    // buffer q, read two groups before its steps: a stage's first two while
    // the last two of the stage before it run.  So stage m + 1 is waited for
    // and published half way through stage m, and the slot of stage m - 1,
    // which every wave has used up by then, takes stage m + kCS - 1.
    float wv[4][4], hv[4][4][NT];
    auto read = [&](int slot, auto qc) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
        const float* ws = &s_w[0][0][0] + slot * (kCK * HM_WAVE) + woff;
        const float* hs = &s_h[0][0][0] + slot * (4 * C * kCH) + hoff;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            wv[q][s] = ws[(16 * q + 4 * s) * HM_WAVE];
#pragma unroll
            for (int n = 0; n < NT; ++n) hv[q][s][n] = hs[(BIG ? 16 : 4) * n * kCH + 16 * q + 4 * s];
        }
        __builtin_amdgcn_sched_barrier(0);  // (the reads before the steps they overlap)
    };
    auto steps = [&](auto qc, auto part, int left) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            // (the last, partial stage: both operands +0 past the end; a chain
            // from +0 never reaches -0, so adding +0 changes nothing)
            const bool in = !decltype(part)::value || 16 * q + 4 * s + g < left;
            const double wd = in ? (double)wv[q][s] : 0.0;
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const double hd = in ? (double)hv[q][s][n] : 0.0;
                if constexpr (BIG) acc[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(hd, wd, acc[n], 0, 0, 0);
                else acc[n] = __builtin_amdgcn_mfma_f64_4x4x4f64(hd, wd, acc[n], 0, 0, 0);
            }
        }
    };
    const std::integral_constant<int, 0> q0;
    const std::integral_constant<int, 1> q1;
    const std::integral_constant<int, 2> q2;
    const std::integral_constant<int, 3> q3;
    for (int m = 0; m < kCS - 1 && m < nm; ++m) issue();
    if (nm >= kCS - 1) wait_vmcnt<(kCS - 2) * NI>();
    else wait_vmcnt<0>();
    lds_barrier();
    read(0, q0);
    read(0, q1);
    int slot = 0;
    auto stage = [&](int m, auto part) __attribute__((always_inline)) {
        const int left = decltype(part)::value ? (int)(hidden - (int64_t)m * kCK) : kCK;
        read(slot, q2);
        steps(q0, part, left);
        read(slot, q3);
        steps(q1, part, left);
        const bool more = m + 1 < nm;
        slot = slot + 1 == kCS ? 0 : slot + 1;
        if (more) {
            // stage m + 1 has landed once at most the stages issued after it
            // are in flight
            if (m + kCS - 2 < nm) wait_vmcnt<(kCS - 3) * NI>();
            else wait_vmcnt<0>();
            lds_barrier();
            if (im < nm) issue();
            read(slot, q0);
        }
        steps(q2, part, left);
        if (more) read(slot, q1);
        steps(q3, part, left);
    };
#pragma clang loop unroll(disable)
    for (int m = 0; m < whole; ++m) stage(m, std::false_type{});
    if (whole < nm) stage(whole, std::true_type{});
    // results: 4 x 4 x 4: row lane / 16, column lane % 16 over the four blocks;
    // 16 x 16 x 4: register r holds row lane / 16 + 4 r, column lane % 16
    const int e = e0 + 16 * wave + li;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
        for (int r = 0; r < (BIG ? 4 : 1); ++r) {
            const int64_t t = t0 + (BIG ? 16 * n + g + 4 * r : 4 * n + g);
            double v;
            if constexpr (BIG) v = acc[n][r];
            else v = acc[n];
            if (t < tokens && e < experts) {
                if (!isfinite(v)) hm_status_or(status, HM_STATUS_NONFINITE_SCORE);
                logits[t * experts + e] = (float)v;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// A2 logits for a few tokens (decode, T <= 16), certified parallel form.
// The reference's logit is float(s_n) with s_k = fl(s_{k-1} + p_k) and
// p_k = h_k w_k (exact in double), k ascending: a chain of H dependent
// additions.  Here H is cut into kNB blocks of b = H/kNB.  Block j is summed
// sequentially from +0 (partials l_jm) beside R_j = sum_m |l_jm| and
// Q_j = sum_m |p_jm| (router_partial_kernel, one wave per block, expert
// group and token); then, per logit, the block sums are added sequentially:
// A_0 = 0, A_{j+1} = fl(A_j + B_j), S' = A_kNB, SA = sum_j |A_{j+1}|.
// Each rounding of the reference errs by at most u|s_k| (u = 2^-53), and
// |s_k| <= |A_j| + |l_jm| plus the (bounded) errors of those, so with
// R = sum R_j and P = sum Q_j
//   |s_n - S'| <= u ((b+1) SA + 2R) + u^2 (H (R + SA) + 1.01 (b^2 + H^2) P).
// Float rounding is monotone: if both ends of S' +- (that bound, inflated
// for the rounding of its own evaluation) round to the same float, it is
// the reference's logit.  Otherwise (about one logit in 10^4 - 10^5 for
// random data, and every non-finite case) the lane runs the reference's
// sequential chain.  HM_EXEC_ROUTE_SEQUENTIAL sends every logit there.
//
// R and P enter the bound only linearly, so each block stores its share
//   C_j = (2u + 2u^2 H) R_j + 2.02 u^2 (b^2 + H^2) Q_j
// and the bound is (u (b+1) + 2u^2 H) SA + sum_j C_j, inflated.
// ---------------------------------------------------------------------------
constexpr int kNB = 32;  // K blocks per logit (a multiple of 8)

__device__ __forceinline__ double block_c_term(double rs, double qs, int64_t hidden) {
    const double u = 0x1p-53;
    const double n = (double)hidden, bw = (double)(hidden / kNB);
    return (2.0 * u + 2.0 * u * u * n) * rs + 2.02 * u * u * (bw * bw + n * n) * qs;
}

// Whether the bound settles float(s_n), given the block-sum chain's result
// a, SA (sa) and the sum of the blocks' C_j (sc).
__device__ __forceinline__ bool block_sums_settle(double a, double sa, double sc,
                                                  int64_t hidden) {
    const double u = 0x1p-53;
    const double n = (double)hidden, bw = (double)(hidden / kNB);
    const double infl = 1.0 + 4.0 * n * u;  // the magnitude sums' own rounding
    const double b0 = ((u * (bw + 1.0) + 2.0 * u * u * n) * sa + sc) * infl;
    const double bc = (b0 * (1.0 + 0x1p-40) + u * fabs(a)) * (1.0 + 0x1p-50);
    const double lo = a - bc, hi = a + bc;
    return isfinite(lo) && isfinite(hi) && __float_as_uint((float)lo) == __float_as_uint((float)hi);
}

// part[t][j][e][c], c = 0, 1: B_j, C_j (block-major: a wave's 64 experts of
// one block are 1 KB in a row, written by one store and read by one load of
// the select kernel, each lane's block pair a 16-byte vector);
// grid (kNB, ceil(E/64), T), one wave, lane = expert.  The block's W rows
// (64 experts wide) go to LDS in one burst of 16-byte DMA loads
// (E % 64 == 0, b % 4 == 0, w 16-byte aligned), else per lane.
//
// With norm.gamma the kernel also is A1 RMSNorm (RMSNorm.cpp:65-77; the
// transformer block runs it on the router's input, TransformerBlock.cpp:
// 88-104): every wave of a token forms the row's tree sum of squares,
// brackets the reference's sequential sum by it as rmsnorm_kernel does, and
// normalises the elements of its own K block; an element the bracket does
// not settle makes the wave take the sequential sum itself, which gives the
// reference's value for every element.  The waves of expert group 0 write
// their blocks to norm.x_out.
constexpr int kPK = 64;  // k per LDS chunk of a block

__global__ __launch_bounds__(64) void router_partial_kernel(
    const float* __restrict__ h, const float* __restrict__ w, int hidden, int experts,
    double* __restrict__ part, int32_t* __restrict__ zero_ctr, int n_zero, hm_norm_fold norm) {
    extern __shared__ float s_row[];  // with the norm: the row (hidden floats)
    __shared__ double s_h[kPK];                                        // broadcast reads
    __shared__ __attribute__((aligned(1024))) float s_w[kPK][HM_WAVE];  // [k][lane]
    const int lane = threadIdx.x;
    // completion counters of the later kernels of a fused decode step start
    // at zero (they run after this kernel has finished)
    if (zero_ctr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0)
        for (int i = lane; i < n_zero; i += HM_WAVE) zero_ctr[i] = 0;
    const int j = blockIdx.x, t = blockIdx.z;
    const int e0 = blockIdx.y * HM_WAVE;
    const int e = e0 + lane;
    const bool live = e < experts;
    const int b = hidden / kNB;
    const bool full = experts % HM_WAVE == 0 && b % 4 == 0 && (uintptr_t)w % 16 == 0;
    const int k0 = j * b;
    const float* hrow = h + (int64_t)t * hidden;
    const float* hp = hrow + k0;
    const bool fold = norm.gamma != nullptr;
    // the whole row in one burst of 16-byte loads (at most 16 per lane)
    const bool row4 = hidden % 256 == 0 && hidden <= 16 * 256 && (uintptr_t)h % 16 == 0;
    double inv_lo = 0.0, inv_hi = 0.0, inv_seq = 0.0;
    bool have_seq = false;
    float4 v[16];  // the row (row4): kept for an LDS copy if the sequential sum is needed
    double acc = 0.0, rs = 0.0, qs = 0.0;
    for (int c0 = 0; c0 < b; c0 += kPK) {
        const int kc = min(kPK, b - c0);
        __builtin_amdgcn_wave_barrier();
        // unconditional loads from clamped addresses (a load under a branch
        // is waited for at the branch's end), masked once they are in
        const int lc = min(lane, kc - 1);
        float hv = hp[c0 + lc];
        const float gv = (fold ? norm.gamma + k0 : hp)[c0 + lc];
        if (full) {
            // lane l: row 4i + l/16, floats 4*(l%16) .. +3 of the 64-expert row
            const float* src = w + (int64_t)(k0 + c0 + (lane >> 4)) * experts + e0 + 4 * (lane & 15);
            for (int i = 0; i < kc / 4; ++i) dma16(src + (int64_t)4 * i * experts, &s_w[4 * i][0]);
        }
        if (fold) {
            if (c0 == 0) {
                // the row's squares, in any order (their loads overlap the
                // block's W burst)
                double ss = 0.0;
                if (row4) {
                    const float4* r4 = reinterpret_cast<const float4*>(hrow);
                    const int n4 = hidden >> 8;
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[i] = r4[lane + HM_WAVE * min(i, n4 - 1)];
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const double q = ((double)v[i].x * v[i].x + (double)v[i].y * v[i].y) +
                                         ((double)v[i].z * v[i].z + (double)v[i].w * v[i].w);
                        ss += i < n4 ? q : 0.0;
                    }
                } else {
                    for (int i = lane; i < hidden; i += HM_WAVE) {
                        const float v = hrow[i];
                        ss += (double)v * v;
                        s_row[i] = v;
                    }
                }
                const double s_fast = hm_wave_sum_f64(ss);
                const double d = hm_rms_sum_slack(hidden);
                inv_lo = hm_inv_rms(s_fast * (1.0 + d), (double)hidden, (double)norm.eps);
                inv_hi = hm_inv_rms(s_fast * (1.0 - d), (double)hidden, (double)norm.eps);
            }
            hv = lane < kc ? hv : 0.0f;
            const double g = lane < kc ? (double)gv : 0.0;
            const float a = (float)((double)hv * inv_lo * g);
            const float bb = (float)((double)hv * inv_hi * g);
            if (!have_seq && (norm.force_seq || __any(__float_as_uint(a) != __float_as_uint(bb)))) {
                // the sequential sum over the row's LDS copy (every lane
                // the same, broadcast reads)
                if (row4) {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (i < (hidden >> 8)) reinterpret_cast<float4*>(s_row)[lane + HM_WAVE * i] = v[i];
                }
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                inv_seq = hm_inv_rms(hm_rms_sum_seq(s_row, hidden), (double)hidden, (double)norm.eps);
                have_seq = true;
            }
            hv = have_seq ? (float)((double)hv * inv_seq * g) : a;
            if (blockIdx.y == 0 && lane < kc) norm.x_out[(int64_t)t * hidden + k0 + c0 + lane] = hv;
        }
        s_h[lane] = lane < kc ? (double)hv : 0.0;
        if (full) {
            wait_vmcnt<0>();
        } else {
            for (int i = 0; i < kc; ++i) s_w[i][lane] = live ? w[(int64_t)(k0 + c0 + i) * experts + e] : 0.0f;
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        auto step = [&](double hk, double wd) __attribute__((always_inline)) {
            acc = __builtin_fma(hk, wd, acc);  // == acc + hk * wd (the product is exact)
            rs += fabs(acc);
            qs = __builtin_fma(fabs(hk), fabs(wd), qs);
        };
        if (kc == kPK) {
            // a whole chunk: the LDS values of the next kRSub steps are read
            // while the current ones are chained, so the chain does not wait
            // for an LDS read every other step (same steps, same order)
            constexpr int kRSub = 16;
            double hb[2][kRSub];
            float wb[2][kRSub];
            auto fetch = [&](int buf, int i0) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < kRSub; ++i) {
                    hb[buf][i] = s_h[i0 + i];
                    wb[buf][i] = s_w[i0 + i][lane];
                }
            };
            fetch(0, 0);
#pragma unroll
            for (int c = 0; c < kPK / kRSub; ++c) {
                if (c + 1 < kPK / kRSub) fetch((c + 1) & 1, (c + 1) * kRSub);
#pragma unroll
                for (int i = 0; i < kRSub; ++i) step(hb[c & 1][i], (double)wb[c & 1][i]);
            }
        } else {
            for (int i = 0; i < kc; ++i) step(s_h[i], (double)s_w[i][lane]);
        }
    }
    if (live) {
        double2* o = reinterpret_cast<double2*>(part + (((int64_t)t * kNB + j) * experts + e) * 2);
        *o = make_double2(acc, block_c_term(rs, qs, hidden));
    }
}

// One logit from its block partials (see above); *settled is false when
// the bound does not settle the float (the caller then runs the sequential
// chain).  pp: this logit's B_0, C_0 (part + (t*kNB*E + e) * 2); block j's
// pair sits 2 E doubles further on per block.
__device__ __forceinline__ float block_logit(const double* __restrict__ pp, int64_t experts,
                                             int64_t hidden, bool force_seq, bool* settled) {
    // all 64 values in 32 vector loads (each block's B_j and C_j in one,
    // so that both sums need every load), then the dependent chain
    typedef int hm_i4 __attribute__((ext_vector_type(4)));
    hm_i4 raw[kNB];
#pragma unroll
    for (int i = 0; i < kNB; ++i) raw[i] = *reinterpret_cast<const hm_i4*>(pp + (int64_t)i * 2 * experts);
    // (every load goes out before the first is used: otherwise the compiler
    // splits each pair and issues the C halves only after the B chain)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kNB; ++i) asm volatile("" : "+v"(raw[i]));
    double a = 0.0, sa = 0.0, sc = 0.0;
#pragma unroll
    for (int i = 0; i < kNB; ++i) {
        const double2 bc = __builtin_bit_cast(double2, raw[i]);
        a += bc.x;
        sa += fabs(a);
        sc += bc.y;
    }
    *settled = !force_seq && block_sums_settle(a, sa, sc, hidden);
    return (float)a;
}

// The reference's sequential chain s_k = fl(s_{k-1} + h_k w_k) (the
// product is exact in double, so fl(s + p) = fma(h, w, s)) for the logit of
// expert e0 + lane of every lane whose bit is set in `need`, four logits at a
// time, one on each 16-lane row (hm_chain64; the operands D chunks of 64
// ahead of the chains: a chunk's W column is 64 cache lines, and its chain
// steps take 160 ns; terms past the end are +0, which leaves every s_k as it
// is: a chain from +0 never reaches -0).  Returns the owning lane's float
// logit (others: v unchanged).
template <int D>
__device__ __forceinline__ float chain_logits(unsigned long long need, int lane, float v, int64_t e0,
                                              const float* __restrict__ hrow,
                                              const float* __restrict__ w, int64_t hidden,
                                              int64_t experts, int32_t* status) {
    while (need) {
        // row r takes the r-th needed logit (the last one again past the end)
        unsigned long long m = need;
        int owner = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = __ffsll((long long)m) - 1;
            if (r <= (lane >> 4)) owner = o;
            if (m & (m - 1)) m &= m - 1;
        }
        const float* wc = w + e0 + owner;
        const int64_t i = 4 * (lane & 15);
        float hv[D][4], wv[D][4];
        auto load = [&](int64_t k0, int d) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t k = min(k0 + i + q, hidden - 1);
                hv[d][q] = hrow[k];
                wv[d][q] = wc[k * experts];
            }
        };
#pragma unroll
        for (int d = 0; d < D; ++d) load(64 * d, d);
        double acc = 0.0;
        for (int64_t k0 = 0; k0 < hidden; k0 += 64 * D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int64_t k = k0 + 64 * d;
                double p[4];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    p[q] = k + i + q < hidden ? (double)hv[d][q] * (double)wv[d][q] : 0.0;
                load(k + 64 * D, d);
                hm_chain64(acc, p[0], p[1], p[2], p[3]);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (!need) break;
            const int o = __ffsll((long long)need) - 1;
            need &= need - 1;
            const double a = __shfl(acc, 16 * r, HM_WAVE);
            if (lane == o) {
                if (!isfinite(a)) hm_status_or(status, HM_STATUS_NONFINITE_SCORE);
                v = (float)a;
            }
        }
    }
    return v;
}

// ---------------------------------------------------------------------------
// A2 select (src/router/CpuRouterBackend.cpp:50-89), one wave per token.
//   softmax: m = max logit; p = expf(l - m) (float, glibc-exact hm_expf);
//            den = sum_e double(p) in ascending e; p = float(double(p)/den).
//   The sum: every p is in [0, 1] and p(max) = 1, so den < 2^12 for
//   E <= 2048.  If every nonzero p is >= 2^-17 its last bit is >= 2^-40,
//   every partial sum is a multiple of 2^-40 below 2^13 and hence exact in
//   double, so any order gives the sequential result; otherwise lane 0 sums
//   sequentially.
//   top-k: k rounds of a wave argmax (hm_rank_key, then the lowest id),
//   i.e. std::partial_sort with the reference comparator.
//   renorm: sum of the k selected scores in rank order in double.
// Writes ids/scores [t, r] in rank order.
// ---------------------------------------------------------------------------
// Softmax, top-k and renormalisation of one token's logits v (one wave; lane
// holds experts lane + 64 j); writes ids/scores [t, r] in rank order.
// A token whose selection failed (the status word says so): placeholder ids
// 0..top_k-1 with zero scores, so that the permutation and expert stages that
// follow on the stream stay in range.
// A token's id and score stores; `coherent`: device-scope stores (sc1,
// written through to the device's coherence point), for a workgroup of
// another XCD that reads them once this one has arrived at the completion
// counter (no L2 write-back needed).
template <typename V>
__device__ __forceinline__ void hm_store_pair(V* p, V v, bool coherent) {
    if (coherent) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
template <typename V>
__device__ __forceinline__ V hm_load_pair(const V* p, bool coherent) {
    return coherent ? __hip_atomic_load(const_cast<V*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                    : *p;
}

__device__ __forceinline__ void select_failed(int lane, int64_t t, int32_t top_k,
                                              uint32_t* __restrict__ ids,
                                              float* __restrict__ scores,
                                              uint32_t* l_ids = nullptr,
                                              float* l_scores = nullptr, bool coherent = false) {
    if (lane < top_k) {
        hm_store_pair(&ids[t * top_k + lane], (uint32_t)lane, coherent);
        hm_store_pair(&scores[t * top_k + lane], 0.0f, coherent);
        if (l_ids) {
            l_ids[lane] = (uint32_t)lane;
            l_scores[lane] = 0.0f;
        }
    }
}

template <int EPL>
__device__ __forceinline__ void select_token(float (&v)[EPL], const bool (&valid)[EPL], int lane,
                                             int wave, int64_t t, int64_t experts, int32_t top_k,
                                             uint32_t flags, uint32_t* __restrict__ ids,
                                             float* __restrict__ scores, int32_t* status,
                                             float* seq_lds, uint32_t* l_ids = nullptr,
                                             float* l_scores = nullptr, bool coherent = false,
                                             const unsigned long long* exp2 = kHmExp2Table) {
    // (l_ids, l_scores: optional LDS copies of this token's ids and scores;
    // coherent: device-scope stores, hm_store_pair; exp2: the expf table,
    // where the caller has it in LDS)
    if (flags & HM_ROUTE_SOFTMAX) {
        float m = -__uint_as_float(0x7f800000u);
#pragma unroll
        for (int j = 0; j < EPL; ++j) if (valid[j]) m = fmaxf(m, v[j]);
        m = hm_wave_max_dpp(m);
        bool exact = true;
        double part = 0.0;
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            if (!valid[j]) continue;
            v[j] = hm_expf_t(__fsub_rn(v[j], m), exp2);
            exact = exact && (v[j] == 0.0f || v[j] >= 0x1p-17f);
            part += (double)v[j];
        }
        double den;
        if (__all(exact) && experts <= 2048) {
            den = hm_wave_sum_f64_dpp(part);
        } else {
            float* seq = seq_lds + (int64_t)wave * experts;
#pragma unroll
            for (int j = 0; j < EPL; ++j) if (valid[j]) seq[lane + HM_WAVE * j] = v[j];
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            double s = 0.0;
            if (lane == 0) for (int64_t e = 0; e < experts; ++e) s += (double)seq[e];
            den = __shfl(s, 0, HM_WAVE);
        }
        if (!(isfinite(den) && den > 0.0)) {
            if (lane == 0) hm_status_or(status, HM_STATUS_SOFTMAX_FAILED);
            select_failed(lane, t, top_k, ids, scores, l_ids, l_scores, coherent);
            return;
        }
#pragma unroll
        for (int j = 0; j < EPL; ++j) if (valid[j]) v[j] = (float)((double)v[j] / den);
    }
    // k rounds of the wave maximum over the scores' order keys; of the lanes
    // that hold it, the lowest expert id still in the running wins (experts
    // lane + 64 j: the first j with such a lane, its lowest lane).  Lane r
    // keeps the r-th id, and after the rounds fetches its score from the lane
    // that holds it.  (32-bit maxima and ballots: a round is a third of the
    // instructions of one over 64-bit (score, id) keys.)
    unsigned key[EPL];
    unsigned long long left[EPL];  // experts not yet taken, by lane
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        key[j] = valid[j] ? hm_rank_key(v[j]) : 0u;
        left[j] = __ballot(valid[j]);
    }
    uint32_t my_id = 0;
    for (int r = 0; r < top_k; ++r) {
        unsigned best = 0u;
#pragma unroll
        for (int j = 0; j < EPL; ++j) best = max(best, key[j]);
        best = hm_wave_max_u32(best);
        unsigned id = 0u;
        bool found = false;
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            const unsigned long long m = __ballot(key[j] == best) & left[j];
            const bool here = !found && m != 0ull;
            const int low = here ? __ffsll((long long)m) - 1 : HM_WAVE;
            id = here ? (unsigned)(HM_WAVE * j + low) : id;
            found = found || here;
            left[j] &= here ? ~(1ull << low) : ~0ull;
            key[j] = lane == low ? 0u : key[j];
        }
        if (lane == r) my_id = id;
    }
    float my_score = 0.0f;
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const float c = __shfl(v[j], (int)(my_id % HM_WAVE), HM_WAVE);
        if ((int)(my_id / HM_WAVE) == j) my_score = c;
    }
    double sel_sum = 0.0;  // rank order, uniform across lanes
    for (int r = 0; r < top_k; ++r)
        sel_sum += (double)__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_score), r));
    if (flags & HM_ROUTE_RENORM) {
        if (!(isfinite(sel_sum) && sel_sum != 0.0)) {
            if (lane == 0) hm_status_or(status, HM_STATUS_RENORM_FAILED);
            select_failed(lane, t, top_k, ids, scores, l_ids, l_scores, coherent);
            return;
        }
        my_score = (float)((double)my_score / sel_sum);
    }
    if (lane < top_k) {
        hm_store_pair(&ids[t * top_k + lane], my_id, coherent);
        hm_store_pair(&scores[t * top_k + lane], my_score, coherent);
        if (l_ids) {
            l_ids[lane] = my_id;
            l_scores[lane] = my_score;
        }
    }
}

// Token t's row in the fixed-point digits of the INT8 expert GEMMs (one wave).
__device__ __forceinline__ void quantize_token(const float* __restrict__ h, int64_t t,
                                               int64_t hidden, int64_t tokens,
                                               const hm_row_quant& xq) {
    const int nv = (int)(hidden / 256);
    const hm_dlay lay = hm_dlay_x(xq.limbs, hidden);
    int8_t* d = xq.digits + t * lay.row;
    int32_t* ds = xq.dsum ? xq.dsum + t : nullptr;
    const float* row = h + t * hidden;
    switch (xq.limbs) {
    case 1: hm_quantize_row_wave<1>(row, nv, d, lay, xq.scales + t, ds, tokens); break;
    case 2: hm_quantize_row_wave<2>(row, nv, d, lay, xq.scales + t, ds, tokens); break;
    default: hm_quantize_row_wave<3>(row, nv, d, lay, xq.scales + t, ds, tokens); break;
    }
}

// Workgroups 0 .. sel-1 select, four tokens each; the others (xq.digits) cut
// four tokens' rows into the fixed-point digits of the INT8 expert GEMMs (the
// block's activation quantisation, one launch fewer).  Both are chains of
// latencies of one wave per token (loads, reductions), so they run side by side
// on waves of their own, and expf's table is read from LDS rather than by a
// gather that waits on memory once per token.  Against one wave doing both in
// turn (128 experts, top-8, H = 2048, three digits): 61 tokens 10 -> 5.7 us,
// 333 11.5 -> 7.3, 2048 15 -> 12; 4096 tokens 19 both ways, where the 84 MB of
// rows read and digits written (16 us at the copy rate) bound it.
template <int EPL>
__global__ __launch_bounds__(kBlock) void router_select_kernel(
    const float* __restrict__ logits, int64_t tokens, int64_t experts,
    int32_t top_k, uint32_t flags, uint32_t* __restrict__ ids,
    float* __restrict__ scores, int32_t* status, const float* __restrict__ h, int64_t hidden,
    hm_row_quant xq, int32_t* __restrict__ hist, unsigned sel) {
    extern __shared__ float seq_lds[];  // (kBlock/64) * experts floats
    __shared__ unsigned long long s_exp2[32];
    const int lane = threadIdx.x & (HM_WAVE - 1);
    const int wave = threadIdx.x / HM_WAVE;
    if (blockIdx.x >= sel) {
        const int64_t t = (int64_t)(blockIdx.x - sel) * (kBlock / HM_WAVE) + wave;
        if (t >= tokens) return;
        quantize_token(h, t, hidden, tokens, xq);
        return;
    }
    const int64_t t = (int64_t)blockIdx.x * (kBlock / HM_WAVE) + wave;
    const float* lt = logits + min(t, tokens - 1) * experts;
    float v[EPL];
    bool valid[EPL];
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const int64_t e = lane + (int64_t)HM_WAVE * j;
        valid[j] = e < experts;
        v[j] = lt[valid[j] ? e : experts - 1];
    }
    hm_load_exp2_table(s_exp2);
    __syncthreads();
    if (t >= tokens) return;
#pragma unroll
    for (int j = 0; j < EPL; ++j) v[j] = valid[j] ? v[j] : 0.0f;
    select_token<EPL>(v, valid, lane, wave, t, experts, top_k, flags, ids, scores, status, seq_lds,
                      nullptr, nullptr, false, s_exp2);
    // The permutation's histogram of each 1024-pair chunk (hm_permute's
    // count pass): each lane re-reads the id it has just written.  Integer
    // counts, so the atomics' order does not matter.
    if (hist && lane < top_k) {
        const int64_t pr = t * top_k + lane;
        atomicAdd(&hist[(pr / kPermChunk) * experts + ids[pr]], 1);
    }
}

// The stable counting sort of permute_count/scatter for at most
// kSmallPairs pairs, by one workgroup (NT threads): counts and offsets
// from an LDS histogram and a block scan, each pair's rank among the
// earlier pairs of its expert by a scan of the ids in LDS.  Ids past the
// expert count (left behind by a routing failure the status word reports)
// are treated as the last expert so that every position stays in range.
constexpr int kSmallPairs = 1024;

template <int NT>
__device__ void permute_small(const uint32_t* __restrict__ ids, const float* __restrict__ scores,
                              int pairs, int top_k, int experts, int32_t* __restrict__ counts,
                              int32_t* __restrict__ offsets, int32_t* __restrict__ perm_tokens,
                              float* __restrict__ perm_weights, int32_t* __restrict__ slots,
                              bool coherent = false) {
    // (coherent: ids and scores read device-scope, hm_load_pair)
    constexpr int EPT = 1024 / NT;  // experts per thread in the scan (E <= 1024)
    __shared__ int s_cnt[1024];
    __shared__ int s_off[1024];
    __shared__ __attribute__((aligned(16))) int s_ids[kSmallPairs];
    __shared__ float s_sc[kSmallPairs];
    __shared__ int s_wsum[NT / HM_WAVE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < experts; i += NT) s_cnt[i] = 0;
    __syncthreads();
    for (int p = tid; p < pairs; p += NT) {
        const uint32_t e = hm_load_pair(&ids[p], coherent);
        s_sc[p] = hm_load_pair(&scores[p], coherent);
        const int ec = e < (uint32_t)experts ? (int)e : experts - 1;
        s_ids[p] = ec;
        atomicAdd(&s_cnt[ec], 1);
    }
    __syncthreads();
    // exclusive scan over experts: thread tid owns experts EPT*tid .. +EPT-1
    int v[EPT], tot = 0;
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int e = EPT * tid + q;
        v[q] = e < experts ? s_cnt[e] : 0;
        tot += v[q];
    }
    int incl = tot;
#pragma unroll
    for (int sft = 1; sft < 64; sft <<= 1) {
        const int o = __shfl_up(incl, sft, 64);
        if (lane >= sft) incl += o;
    }
    if (lane == 63) s_wsum[wave] = incl;
    __syncthreads();
    int base = incl - tot;
    for (int wv = 0; wv < wave; ++wv) base += s_wsum[wv];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int e = EPT * tid + q;
        if (e < experts) {
            s_off[e] = base;
            counts[e] = v[q];
            offsets[e] = base;
            if (e == experts - 1) offsets[experts] = base + v[q];
        }
        base += v[q];
    }
    __syncthreads();
    // 64 pairs a wave at a time: a pair's rank in its group is the number of
    // earlier pairs with its id, those of the same 64 from one ballot per id
    // bit, those before them four to an LDS read
    for (int c = wave; c * HM_WAVE < pairs; c += NT / HM_WAVE) {
        const int p = c * HM_WAVE + lane;
        const bool live = p < pairs;
        const int e = s_ids[live ? p : pairs - 1];
        unsigned long long same = __ballot(live);
        for (int b = 0; (1 << b) < experts; ++b) {
            const bool bit = (e >> b) & 1;
            const unsigned long long m = __ballot(bit);
            same &= bit ? m : ~m;
        }
        int rank = __popcll(same & ((1ull << lane) - 1));
        const int4* s4 = reinterpret_cast<const int4*>(s_ids);
#pragma unroll 4
        for (int q = 0; q < c * (HM_WAVE / 4); ++q) {
            const int4 x = s4[q];
            rank += (x.x == e) + (x.y == e) + (x.z == e) + (x.w == e);
        }
        if (live) {
            const int pos = s_off[e] + rank;
            perm_tokens[pos] = p / top_k;
            perm_weights[pos] = s_sc[p];
            slots[p] = pos;
        }
    }
}

// The grouping of permute_small for P <= 64 pairs by one wave, in
// registers: lane p holds pair p (its id, clamped to the expert count as
// permute_small does, and score); its position is the number of pairs with
// a smaller expert plus the earlier pairs of its own expert (the stable
// counting sort), the lanes' experts lane + 64 j count their pairs and
// those of smaller experts (counts, offsets), each pair's id read in turn
// across the wave.
template <int EPL>
__device__ __forceinline__ void permute_wave(uint32_t id, float score, int pairs, int top_k,
                                             int experts, int32_t* __restrict__ counts,
                                             int32_t* __restrict__ offsets,
                                             int32_t* __restrict__ perm_tokens,
                                             float* __restrict__ perm_weights,
                                             int32_t* __restrict__ slots) {
    const int lane = threadIdx.x & (HM_WAVE - 1);
    const int ep = lane < pairs ? (int)min(id, (uint32_t)(experts - 1)) : INT_MAX;
    int less = 0, same = 0;
    int cnt[EPL], off[EPL];
#pragma unroll
    for (int j = 0; j < EPL; ++j) cnt[j] = off[j] = 0;
    for (int q = 0; q < pairs; ++q) {
        const int eq = __builtin_amdgcn_readlane(ep, q);
        less += eq < ep;
        same += (eq == ep) & (q < lane);
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            const int e = lane + HM_WAVE * j;
            cnt[j] += eq == e;
            off[j] += eq < e;
        }
    }
    if (lane < pairs) {
        const int pos = less + same;
        perm_tokens[pos] = lane / top_k;
        perm_weights[pos] = score;
        slots[lane] = pos;
    }
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const int e = lane + HM_WAVE * j;
        if (e < experts) {
            counts[e] = cnt[j];
            offsets[e] = off[j];
            if (e == experts - 1) offsets[experts] = off[j] + cnt[j];
        }
    }
}

// Select over logits formed from the decode partials (and written to
// `logits` too).  !SPLIT: NW tokens per workgroup, one per wave.  SPLIT: one
// token per workgroup, its rows of 64 logits shared out over the NW waves
// so that all their loads are in flight together (each token reads 2 kNB
// doubles per logit, 64 KB at E = 128, that other CUs wrote), wave 0
// selecting.  With PERMUTE the workgroup that finishes last (a device
// counter, zeroed by router_partial_kernel) also sorts the pairs into
// expert groups, which is hm_permute's result: one launch fewer per decode
// step; a single workgroup hands its ids and scores over in LDS.  With
// xq.digits a second set of workgroups cuts the tokens' rows into digits
// beside the selecting ones.  All of it is latency of one wave per token and
// of the last workgroup's grouping; ranks from ballots (a loop over the
// earlier pairs before), 32-bit argmax rounds (64-bit keys before), expf's
// table in LDS and the digits on workgroups of their own took it from 12.0 to
// 9.8 us at 16 tokens, 128 experts, and 13.2 to 10.6 at 64 experts in FP32.
template <int EPL, bool PERMUTE, int NW, bool SPLIT>
__global__ __launch_bounds__(NW * HM_WAVE) void router_select_partial_kernel(
    const float* __restrict__ h, const float* __restrict__ w, const double* __restrict__ part,
    int64_t tokens, int64_t hidden, int64_t experts, int32_t top_k, uint32_t flags,
    float* __restrict__ logits, uint32_t* __restrict__ ids, float* __restrict__ scores,
    int32_t* status, int32_t* __restrict__ done_ctr, int32_t* __restrict__ counts,
    int32_t* __restrict__ offsets, int32_t* __restrict__ perm_tokens,
    float* __restrict__ perm_weights, int32_t* __restrict__ slots, hm_row_quant xq) {
    extern __shared__ float seq_lds[];  // NW * experts floats
    // one workgroup: the grouping reads the ids and scores from LDS copies
    __shared__ uint32_t s_sel_ids[PERMUTE ? NW * 64 : 1];
    __shared__ float s_sel_sc[PERMUTE ? NW * 64 : 1];
    // SPLIT: the token's logits, rows of 64 experts shared out over the waves
    __shared__ float s_lg[SPLIT ? EPL : 1][HM_WAVE];
    if (SPLIT && blockIdx.x >= tokens) {
        if (threadIdx.x < HM_WAVE) quantize_token(h, blockIdx.x - tokens, hidden, tokens, xq);
        return;
    }
    // expf's table: its load goes out before the partials' and its LDS copy
    // is written once they are in
    __shared__ unsigned long long s_exp2[32];
    const unsigned long long exp2 = kHmExp2Table[threadIdx.x & 31];
    const bool local = PERMUTE && tokens == 1;
    // several workgroups: the last to arrive groups every token's pairs, so
    // the ids and scores go out device-coherent
    const bool shared = PERMUTE && tokens > 1;
    const int lane = threadIdx.x & (HM_WAVE - 1);
    const int wave = threadIdx.x / HM_WAVE;
    const bool force_seq = (flags & HM_EXEC_ROUTE_SEQUENTIAL) != 0;
    // one logit row j (experts 64 j + lane) of token t: its block sums, and
    // the reference's chain where the bound leaves it open
    auto logit_row = [&](int64_t t, int j, bool& valid) __attribute__((always_inline)) -> float {
        const int64_t e = lane + (int64_t)HM_WAVE * j;
        valid = e < experts;
        bool settled;
        // (lanes past the experts read the last expert's: no branch around the loads)
        float v = block_logit(part + (t * kNB * experts + (valid ? e : experts - 1)) * 2, experts,
                              hidden, force_seq, &settled);
        if (!valid) {
            v = 0.0f;
            settled = true;
        }
        v = chain_logits<4>(__ballot(valid && !settled), lane, v, (int64_t)HM_WAVE * j,
                         h + t * hidden, w, hidden, experts, status);
        if (valid) logits[t * experts + e] = v;
        return v;
    };
    if constexpr (SPLIT) {
        // one token per workgroup: wave w forms rows w, w + NW, .., so that
        // every row's loads are in flight at once; wave 0 selects
        const int64_t t = blockIdx.x;
        for (int j = wave; j < EPL; j += NW) {
            bool valid;
            s_lg[j][lane] = logit_row(t, j, valid);
        }
        if (threadIdx.x < 32) s_exp2[threadIdx.x] = exp2;
        __syncthreads();
        if (wave == 0) {
            float v[EPL];
            bool valid[EPL];
#pragma unroll
            for (int j = 0; j < EPL; ++j) {
                v[j] = s_lg[j][lane];
                valid[j] = lane + (int64_t)HM_WAVE * j < experts;
            }
            select_token<EPL>(v, valid, lane, 0, t, experts, top_k, flags, ids, scores, status,
                              seq_lds, local ? s_sel_ids : nullptr, local ? s_sel_sc : nullptr,
                              shared, s_exp2);
            if (local && top_k <= HM_WAVE) {
                // one token: its grouping by this wave, from the LDS copies
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                const int ln = lane < top_k ? lane : 0;
                permute_wave<EPL>(s_sel_ids[ln], s_sel_sc[ln], top_k, top_k, (int)experts,
                                  counts, offsets, perm_tokens, perm_weights, slots);
            }
        }
        if (local && top_k <= HM_WAVE) return;
    } else {
        // one token per wave
        const int64_t t = (int64_t)blockIdx.x * NW + wave;
        if (threadIdx.x < 32) s_exp2[threadIdx.x] = exp2;
        __syncthreads();
        if (t < tokens) {
            float v[EPL];
            bool valid[EPL];
#pragma unroll
            for (int j = 0; j < EPL; ++j) v[j] = logit_row(t, j, valid[j]);
            select_token<EPL>(v, valid, lane, wave, t, experts, top_k, flags, ids, scores, status,
                              seq_lds, local ? s_sel_ids + wave * top_k : nullptr,
                              local ? s_sel_sc + wave * top_k : nullptr, shared, s_exp2);
        }
    }
    if constexpr (PERMUTE) {
        if (tokens > 1) {
            // Arrival without a write-back of this XCD's L2: the ids and
            // scores were stored device-coherent (sc1); once this wave's
            // stores are complete (vmcnt 0, every wave) the workgroup counts
            // in, and the last one reads them device-coherent too.
            __shared__ int s_last;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (threadIdx.x == 0)
                s_last = __hip_atomic_fetch_add(done_ctr, 1, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT) == (int)tokens - 1;
            __syncthreads();
            if (!s_last) return;
        } else {
            __syncthreads();  // one workgroup: its own ids and scores
        }
        permute_small<NW * HM_WAVE>(local ? s_sel_ids : ids, local ? s_sel_sc : scores,
                                    (int)(tokens * top_k), top_k, (int)experts, counts, offsets,
                                    perm_tokens, perm_weights, slots, shared);
    }
}

// ---------------------------------------------------------------------------
// One-token decode step: router_select_partial_kernel's select, redone by
// every workgroup of the gate/up slice launch, then that workgroup's slice
// (hm_gemv_slice.h).  One token's select reads 2 kNB doubles per logit
// (64 KB at E = 128) that every XCD's L2 serves to its workgroups, and
// costs a few hundred cycles of FP64 arithmetic: less than the launch it
// replaces.  Workgroup (bx, by): columns 8 bx .. +7 of the by-th selected
// expert in ascending id (its grouped row is by: one token, distinct
// experts).  Workgroup (0, 0) also writes the routing results (logits, ids,
// scores, the groups, the status word) for the down kernel and the caller;
// the others keep theirs in LDS.  Same results as the two kernels it
// replaces: the same functions on the same partials.
// ---------------------------------------------------------------------------
// Workgroup phases: (1) the token row's loads, then every wave loads a
// quarter (E <= 64: an eighth) of one logit row's block partials, all in
// flight at once, and puts the blocks' B_j and its share of sum C_j in LDS;
// (2) wave j forms row j's block-sum chain and bound from LDS (as
// block_logit; the C_j summed in another order, which the bound's
// inflation covers), the reference's chain where the bound leaves a logit
// open; (3) wave 0: softmax, top-k, renormalisation (select_token), the lead
// workgroup writes the results and the groups; (4) the slice.
template <int EPL, int LJ>
__global__ __launch_bounds__(kGvThreads) void select_gateup_kernel(
    const float* __restrict__ h, const float* __restrict__ w, const double* __restrict__ part,
    int64_t hidden, int64_t experts, int32_t top_k, uint32_t flags, float* __restrict__ logits,
    uint32_t* __restrict__ ids, float* __restrict__ scores, int32_t* status,
    int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ perm_tokens, float* __restrict__ perm_weights,
    int32_t* __restrict__ slots, int64_t inter, const int8_t* __restrict__ packed,
    const float* __restrict__ scale, const int32_t* __restrict__ zp, float* __restrict__ z) {
    static_assert(EPL == 1 || EPL == 2, "at most two rows of 64 logits (LDS)");
    constexpr int WPR = kGvWaves / EPL;  // waves per logit row
    constexpr int BPW = kNB / WPR;       // blocks per wave
    typedef int hm_i4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) float s_x[];  // the token row (K32 floats)
    __shared__ double s_b[EPL][kNB][HM_WAVE];
    __shared__ double s_c[EPL][WPR][HM_WAVE];
    __shared__ float s_seq[EPL * HM_WAVE];
    __shared__ float s_lg[EPL][HM_WAVE];
    __shared__ unsigned long long s_exp2[32];
    __shared__ uint32_t s_sel_ids[HM_WAVE], s_own_ids[HM_WAVE];
    __shared__ float s_sel_sc[HM_WAVE], s_own_sc[HM_WAVE];
    const int tid = threadIdx.x, lane = tid & (HM_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool lead = blockIdx.x == 0 && blockIdx.y == 0;
    int32_t* st = lead ? status : nullptr;
    const unsigned long long exp2 = kHmExp2Table[tid & 31];
    // (1) the token row (K = hidden, a multiple of 32: no padding), then the
    // partials of row j, blocks q BPW .. +BPW-1
    const int k4 = (int)(hidden / 4);
    float4 xa[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
        xa[u] = reinterpret_cast<const float4*>(h)[min(tid + u * kGvThreads, k4 - 1)];
    {
        const int j = wave / WPR, q = wave % WPR;
        const int64_t e = lane + (int64_t)HM_WAVE * j;
        const double* pp = part + (e < experts ? e : experts - 1) * 2 +
                           (int64_t)q * BPW * 2 * experts;
        hm_i4 raw[BPW];
#pragma unroll
        for (int i = 0; i < BPW; ++i) raw[i] = *reinterpret_cast<const hm_i4*>(pp + (int64_t)i * 2 * experts);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < BPW; ++i) asm volatile("" : "+v"(raw[i]));
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (tid + u * kGvThreads < k4) reinterpret_cast<float4*>(s_x)[tid + u * kGvThreads] = xa[u];
        double cs = 0.0;
#pragma unroll
        for (int i = 0; i < BPW; ++i) {
            const double2 bc = __builtin_bit_cast(double2, raw[i]);
            s_b[j][q * BPW + i][lane] = bc.x;
            cs += bc.y;
        }
        s_c[j][q][lane] = cs;
    }
    if (tid < 32) s_exp2[tid] = exp2;
    __syncthreads();
    // (2) the logits, row j by wave j
    if (wave < EPL) {
        const int64_t e = lane + (int64_t)HM_WAVE * wave;
        const bool valid = e < experts;
        double a = 0.0, sa = 0.0, sc = 0.0;
#pragma unroll
        for (int i = 0; i < kNB; ++i) {
            a += s_b[wave][i][lane];
            sa += fabs(a);
        }
#pragma unroll
        for (int q = 0; q < WPR; ++q) sc += s_c[wave][q][lane];
        const bool settled = !valid || ((flags & HM_EXEC_ROUTE_SEQUENTIAL) == 0 &&
                                        block_sums_settle(a, sa, sc, hidden));
        float v = valid ? (float)a : 0.0f;
        v = chain_logits<1>(__ballot(valid && !settled), lane, v, (int64_t)HM_WAVE * wave, h, w,
                         hidden, experts, st);
        if (lead && valid) logits[e] = v;
        s_lg[wave][lane] = v;
    }
    __syncthreads();
    // (3) softmax, top-k, renormalisation (wave 0); the lead workgroup
    // writes the results and the groups
    if (wave == 0) {
        float v[EPL];
        bool valid[EPL];
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            v[j] = s_lg[j][lane];
            valid[j] = lane + (int64_t)HM_WAVE * j < experts;
        }
        select_token<EPL>(v, valid, lane, 0, 0, experts, top_k, flags, lead ? ids : s_own_ids,
                          lead ? scores : s_own_sc, st, s_seq, s_sel_ids, s_sel_sc, false, s_exp2);
        if (lead) {
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const int ln = lane < top_k ? lane : 0;
            permute_wave<EPL>(s_sel_ids[ln], s_sel_sc[ln], top_k, top_k, (int)experts, counts,
                              offsets, perm_tokens, perm_weights, slots);
        }
    }
    __syncthreads();
    // (4) this workgroup's expert: the selected id of rank by (ids clamped to
    // the expert count, as the grouping does), and its slice
    const uint32_t my = lane < top_k ? min(s_sel_ids[lane], (uint32_t)(experts - 1)) : 0xffffffffu;
    int rank = 0;
    for (int q = 0; q < top_k; ++q) rank += (uint32_t)__shfl((int)my, q, HM_WAVE) < my;
    const unsigned long long hit = __ballot(lane < top_k && rank == (int)blockIdx.y);
    const int e = hit ? __builtin_amdgcn_readlane((int)my, __ffsll((long long)hit) - 1) : -1;
    gateup_slice_body<1, LJ, true, 1>(blockIdx.x, blockIdx.y,
                                      hm_slice_pre{e, (int)blockIdx.y, 1, 0}, h, nullptr, hidden,
                                      inter, experts, packed, scale, zp, nullptr, 1, z);
}

// ---------------------------------------------------------------------------
// A3 permute (src/router/CpuRouterBackend.cpp:140-159).  The reference
// appends (t, score) to group ids[t,r] walking tokens in ascending order and
// then sorts the groups by id: a stable counting sort of the T*k pairs in
// token-major order.  Here the pairs are cut into chunks of 1024:
//   permute_count_kernel    one workgroup per chunk: the chunk's expert
//                           histogram (LDS, order-free) -> hist[chunk][E]
//   permute_scatter_kernel  one workgroup per chunk: offsets[e] (exclusive
//                           scan of the column sums), the chunk's base per
//                           expert (lower chunks' counts), and each pair's
//                           rank among the chunk's earlier pairs of the same
//                           expert (shuffles inside a wave, per-wave counts
//                           across waves) -> its grouped position.
// No global atomics; every position is a pure function of the ids.  A single
// chunk (decode) needs no histogram pass.
// ---------------------------------------------------------------------------
constexpr int kPermThreads = kPermChunk;
constexpr int kPermWaves = kPermThreads / 64;

// Ids past the expert count (a caller's bad input, or the placeholders a
// failed routing leaves for the status word to report) count as the last
// expert, as in permute_small: every LDS index and grouped position stays in
// range whatever the ids hold.
__device__ __forceinline__ int clamp_expert(uint32_t e, int64_t experts) {
    return e < (uint64_t)experts ? (int)e : (int)experts - 1;
}

__global__ __launch_bounds__(kPermThreads) void permute_count_kernel(
    const uint32_t* __restrict__ ids, int64_t pairs, int64_t experts, int32_t* __restrict__ hist) {
    __shared__ int h[1024];
    const int tid = threadIdx.x;
    for (int i = tid; i < experts; i += kPermThreads) h[i] = 0;
    __syncthreads();
    const int64_t p = (int64_t)blockIdx.x * kPermThreads + tid;
    if (p < pairs) atomicAdd(&h[clamp_expert(ids[p], experts)], 1);
    __syncthreads();
    for (int i = tid; i < experts; i += kPermThreads) hist[(int64_t)blockIdx.x * experts + i] = h[i];
}

__global__ __launch_bounds__(kPermThreads) void permute_scatter_kernel(
    const uint32_t* __restrict__ ids, const float* __restrict__ scores, int64_t pairs,
    int32_t top_k, int64_t experts, const int32_t* __restrict__ hist, int64_t chunks,
    int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ perm_tokens, float* __restrict__ perm_weights,
    int32_t* __restrict__ slots) {
    __shared__ int base[1024];                 // this chunk's first position per expert
    __shared__ int wcount[kPermWaves][1024];   // per-wave counts (this chunk)
    __shared__ int scan_w[kPermWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t c = blockIdx.x;
    const int64_t p = c * kPermThreads + tid;
    const int e = p < pairs ? clamp_expert(ids[p], experts) : -1;
    for (int i = tid; i < kPermWaves * experts; i += kPermThreads)
        wcount[i / experts][i % experts] = 0;
    __syncthreads();
    if (e >= 0) atomicAdd(&wcount[wave][e], 1);
    __syncthreads();
    // column sums over chunks (total per expert) and the lower chunks' part
    int total = 0, before = 0;
    if (tid < experts) {
        if (hist) {
            // (eight loads in flight per round)
            for (int64_t c0 = 0; c0 < chunks; c0 += 8) {
                int v[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) v[q] = c0 + q < chunks ? hist[(c0 + q) * experts + tid] : 0;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    total += v[q];
                    if (c0 + q < c) before += v[q];
                }
            }
        } else {
            for (int w = 0; w < kPermWaves; ++w) total += wcount[w][tid];
        }
    }
    // exclusive scan of the totals over experts (one value per thread)
    int incl = total;
#pragma unroll
    for (int sft = 1; sft < 64; sft <<= 1) {
        const int o = __shfl_up(incl, sft, 64);
        if (lane >= sft) incl += o;
    }
    if (lane == 63) scan_w[wave] = incl;
    __syncthreads();
    int wbase = 0;
    for (int w = 0; w < wave; ++w) wbase += scan_w[w];
    const int offset = wbase + incl - total;
    if (tid < experts) {
        base[tid] = offset + before;
        if (c == 0) {
            counts[tid] = total;
            offsets[tid] = offset;
            if (tid == experts - 1) offsets[experts] = offset + total;
        }
    }
    __syncthreads();
    if (e < 0) return;
    // rank among the chunk's earlier pairs of the same expert: earlier
    // waves' counts, then the wave's earlier lanes with the same id (their
    // mask from one ballot per id bit over the wave's remaining lanes;
    // pairs past the end have left and come after every live pair)
    int rank = 0;
    for (int w = 0; w < wave; ++w) rank += wcount[w][e];
    unsigned long long same = __ballot(true);
    for (int b = 0; (1 << b) < experts; ++b) {
        const bool bit = (e >> b) & 1;
        const unsigned long long m = __ballot(bit);
        same &= bit ? m : ~m;
    }
    rank += __popcll(same & ((1ull << lane) - 1));
    const int pos = base[e] + rank;
    perm_tokens[pos] = (int32_t)(p / top_k);
    perm_weights[pos] = scores[p];
    slots[p] = pos;
}

// A4 gather (MoERuntime.cpp:288-298).
__global__ void gather_rows_kernel(const float* __restrict__ in,
                                   const int32_t* __restrict__ rows,
                                   int64_t count, int64_t width,
                                   float* __restrict__ out) {
    const int64_t r = blockIdx.y;
    const float* src = in + (int64_t)rows[r] * width;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < width;
         i += (int64_t)gridDim.x * kBlock) {
        out[r * width + i] = src[i];
    }
}


// ---------------------------------------------------------------------------
// A7 combine (src/core/runtime/MoERuntime.cpp:312-324): per token, the
// reference adds w * y over groups in ascending expert id, starting from 0,
// with a separate float multiply and add.  The k selected ids of a token are
// distinct, so ranking them gives that order.  One workgroup per token; each
// thread owns 4-element column groups (float4 loads and stores).  Optional
// residual added last (TransformerBlock.cpp:101-104).
// ---------------------------------------------------------------------------
constexpr int kMaxTopK = 64;

__global__ __launch_bounds__(kBlock) void combine_kernel(
    const float* __restrict__ y, const uint32_t* __restrict__ ids,
    const int32_t* __restrict__ slots, const float* __restrict__ scores,
    int64_t tokens, int32_t top_k, int64_t width,
    const float* __restrict__ residual, float* __restrict__ out) {
    __shared__ int64_t srow[kMaxTopK];
    __shared__ float sw[kMaxTopK];
    const int64_t t = blockIdx.x;
    const int tid = threadIdx.x;
    if (tid < top_k) {  // rank of this pair among the token's ids, ascending
        const uint32_t id = ids[t * top_k + tid];
        int rank = 0;
        for (int r = 0; r < top_k; ++r) rank += ids[t * top_k + r] < id;
        srow[rank] = slots[t * top_k + tid];
        sw[rank] = scores[t * top_k + tid];
    }
    __syncthreads();
    if ((width & 3) == 0) {
        const int64_t w4 = width >> 2;
        // two column groups per thread per pass: sixteen rows' float4 loads
        // in flight before the adds (ascending order per column); y is read
        // once, with the streaming hint
        for (int64_t i0 = tid; i0 < w4; i0 += 2 * kBlock) {
          float4 res[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) res[h] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          for (int r0 = 0; r0 < top_k; r0 += 8) {
            float4 v[2][8];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int64_t i = i0 + h * kBlock;
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    v[h][q] = r0 + q < top_k && i < w4
                                  ? hm_load_stream(
                                        reinterpret_cast<const float4*>(y + srow[r0 + q] * width) + i)
                                  : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float4 acc = res[h];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    if (r0 + q < top_k) {
                        const float wv = sw[r0 + q];
                        acc.x = __fadd_rn(acc.x, __fmul_rn(wv, v[h][q].x));
                        acc.y = __fadd_rn(acc.y, __fmul_rn(wv, v[h][q].y));
                        acc.z = __fadd_rn(acc.z, __fmul_rn(wv, v[h][q].z));
                        acc.w = __fadd_rn(acc.w, __fmul_rn(wv, v[h][q].w));
                    }
                }
                res[h] = acc;
            }
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int64_t i = i0 + h * kBlock;
            if (i >= w4) break;
            float4 acc = res[h];
            if (residual) {
                const float4 rv = reinterpret_cast<const float4*>(residual + t * width)[i];
                acc.x = __fadd_rn(rv.x, acc.x);
                acc.y = __fadd_rn(rv.y, acc.y);
                acc.z = __fadd_rn(rv.z, acc.z);
                acc.w = __fadd_rn(rv.w, acc.w);
            }
            reinterpret_cast<float4*>(out + t * width)[i] = acc;
          }
        }
        return;
    }
    for (int64_t i = tid; i < width; i += kBlock) {
        float acc = 0.0f;
        for (int r = 0; r < top_k; ++r) acc = __fadd_rn(acc, __fmul_rn(sw[r], y[srow[r] * width + i]));
        if (residual) acc = __fadd_rn(residual[t * width + i], acc);
        out[t * width + i] = acc;
    }
}

// A6 elementwise (Activation.cpp:44, CpuTensorBackend.cpp:202-204, 217-219).
__global__ void silu_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) y[i] = hm_silu(x[i]);
}
__global__ void mul_kernel(const float* __restrict__ a, const float* __restrict__ b,
                           float* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) y[i] = __fmul_rn(a[i], b[i]);
}
__global__ void add_kernel(const float* __restrict__ a, const float* __restrict__ b,
                           float* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) y[i] = __fadd_rn(a[i], b[i]);
}
__global__ void expf_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) y[i] = hm_expf(x[i]);
}

unsigned grid_for(int64_t n) {
    int64_t g = (n + kBlock - 1) / kBlock;
    if (g < 1) g = 1;
    if (g > 65535) g = 65535;
    return (unsigned)g;
}


}  // namespace

// hm_rmsnorm's launch; force_seq: every row takes the sequential sum of
// squares (HM_EXEC_ROUTE_SEQUENTIAL through hm_moe_layer_forward).
int hm_launch_rmsnorm(const float* x, const float* gamma, float* y, int64_t rows,
                      int64_t width, float eps, bool force_seq, void* stream) {
    HM_REQUIRE(x && gamma && y && rows >= 0 && width > 0);
    HM_REQUIRE(std::isfinite(eps) && eps > 0.0f);  // RMSNorm.cpp:22
    HM_REQUIRE(width <= 16384);                     // row staged in LDS
    if (rows == 0) return HM_OK;
    HM_REQUIRE(rows <= INT_MAX);
    const bool aligned = ((uintptr_t)x | (uintptr_t)gamma | (uintptr_t)y) % 16 == 0;
    if (aligned && width % 256 == 0 && width / 256 <= 16) {
        const unsigned grid = (unsigned)((rows + kBlock / HM_WAVE - 1) / (kBlock / HM_WAVE));
        const hipStream_t s = hm_stream(stream);
        const int fs = force_seq ? 1 : 0;
        switch (width / 256) {
#define HM_RMS_CASE(v) \
    case v: hipLaunchKernelGGL(rmsnorm_wave_kernel<v>, dim3(grid), dim3(kBlock), 0, s, x, gamma, y, rows, eps, fs); break;
            HM_RMS_CASE(1) HM_RMS_CASE(2) HM_RMS_CASE(3) HM_RMS_CASE(4) HM_RMS_CASE(5) HM_RMS_CASE(6)
            HM_RMS_CASE(7) HM_RMS_CASE(8) HM_RMS_CASE(9) HM_RMS_CASE(10) HM_RMS_CASE(11)
            HM_RMS_CASE(12) HM_RMS_CASE(13) HM_RMS_CASE(14) HM_RMS_CASE(15) HM_RMS_CASE(16)
#undef HM_RMS_CASE
        }
        HM_LAUNCHED();
        return HM_OK;
    }
    hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)rows), dim3(kBlock),
                       (size_t)width * sizeof(float), hm_stream(stream), x, gamma,
                       y, width, eps, force_seq ? 1 : 0);
    HM_LAUNCHED();
    return HM_OK;
}

extern "C" {

int hm_rmsnorm(const float* x, const float* gamma, float* y, int64_t rows,
               int64_t width, float eps, void* stream) {
    return hm_launch_rmsnorm(x, gamma, y, rows, width, eps, false, stream);
}


// Route workspace: the logits [T x E] floats (rounded up to 256 bytes), then
// for decode batches (T <= kDecodeTokens) the block partials
// [T x E x 2 x kNB] doubles.
constexpr int64_t kDecodeTokens = 16;

static size_t route_logits_bytes(int64_t tokens, int64_t experts) {
    return ((size_t)tokens * (size_t)experts * sizeof(float) + 255) & ~(size_t)255;
}

// The bytes a caller provides.  A batch with E % 64 == 0 is asked for 8-byte
// sums of up to eight K ranges, both operands' norms and a copy of W beside the
// logits, which it no longer fills: the size is part of the interface (callers
// allocate by it, and the block without allocation accepts batches by it).
size_t hm_route_workspace_bytes(int64_t tokens, int64_t hidden, int64_t experts) {
    if (tokens < 0 || experts <= 0 || hidden <= 0) return 0;
    if (tokens > kDecodeTokens) {
        size_t b = route_logits_bytes(tokens, experts);
        if (experts % HM_WAVE == 0) {
            const int64_t tiles = ((tokens + 63) / 64) * (experts / HM_WAVE);
            size_t sp = 1;
            while (sp < 8 && tiles * (int64_t)sp < 512) sp *= 2;
            b += sp * ((size_t)tokens * (size_t)experts + (size_t)tokens + (size_t)experts) *
                     sizeof(double) +
                 (size_t)experts * (size_t)hidden * sizeof(float);
        }
        return b;
    }
    return route_logits_bytes(tokens, experts) +
           (size_t)tokens * (size_t)experts * kNB * 2 * sizeof(double);
}

}  // extern "C"

// The logits of a batch (router_chain_kernel); hc: the permutation's chunk
// histograms to clear.
static int launch_router_chains(const float* h, const float* w, int64_t tokens, int64_t hidden,
                                int64_t experts, float* logits, int32_t* status, int32_t* hc,
                                int hc_n, void* stream) {
    const int64_t eb = (experts + HM_WAVE - 1) / HM_WAVE;
    // 4 C tokens a workgroup: the shortest rounds of workgroups (above
    // router_chain_kernel)
    const int chains[4] = {1, 2, 4, 8};
    const double cost[4] = {17.0, 24.0, 29.0, 46.0};
    int c = 1;
    double best = 0.0;
    for (int i = 0; i < 4; ++i) {
        const int64_t wgs = (tokens + 4 * chains[i] - 1) / (4 * chains[i]) * eb;
        const double us = (double)((wgs + 255) / 256) * cost[i];
        if (i == 0 || us < best) {
            best = us;
            c = chains[i];
        }
    }
    const dim3 grid((unsigned)((tokens + 4 * c - 1) / (4 * c)), (unsigned)eb);
    const bool vec = experts % HM_WAVE == 0 && (uintptr_t)w % 16 == 0;
#define HM_CHAINS(C)                                                                            \
    do {                                                                                        \
        if (vec)                                                                                \
            hipLaunchKernelGGL((router_chain_kernel<C, true>), grid, dim3(256), 0, hm_stream(stream), \
                               h, w, tokens, hidden, (int)experts, logits, status, hc, hc_n);   \
        else                                                                                    \
            hipLaunchKernelGGL((router_chain_kernel<C, false>), grid, dim3(256), 0, hm_stream(stream), \
                               h, w, tokens, hidden, (int)experts, logits, status, hc, hc_n);   \
    } while (0)
    if (c == 1) HM_CHAINS(1);
    else if (c == 2) HM_CHAINS(2);
    else if (c == 4) HM_CHAINS(4);
    else HM_CHAINS(8);
#undef HM_CHAINS
    HM_LAUNCHED();
    return HM_OK;
}

// The decode router's two launches.  With `fused`, the select kernel also
// forms the expert groups (the workgroup that finishes last) and the
// partial kernel zeroes the fused step's completion counters first.
static int launch_decode_router(const float* h, const float* w, int64_t tokens, int64_t hidden,
                                int64_t experts, int32_t top_k, uint32_t flags, float* logits,
                                uint32_t* ids, float* scores, int32_t* status, void* route_ws,
                                const hm_decode_fusion* fused, const hm_norm_fold* norm,
                                const hm_row_quant* xq, void* stream, bool select = true) {
    const hm_row_quant q = xq && fused ? *xq : hm_row_quant{nullptr, nullptr, nullptr, 0};
    const int epl = (int)((experts + HM_WAVE - 1) / HM_WAVE);
    // fused: one token per workgroup, its logit rows shared out over up to
    // four waves; else four tokens (waves) per workgroup
    const int nw = !fused ? 4 : epl <= 1 ? 1 : epl <= 2 ? 2 : 4;
    const dim3 sgrid((unsigned)(fused ? (q.digits ? 2 * tokens : tokens) : (tokens + 3) / 4));
    const size_t seq_bytes = (size_t)nw * experts * sizeof(float);
    double* part = reinterpret_cast<double*>(static_cast<char*>(route_ws) +
                                             route_logits_bytes(tokens, experts));
    const dim3 pgrid((unsigned)kNB, (unsigned)((experts + HM_WAVE - 1) / HM_WAVE),
                     (unsigned)tokens);
    const hm_norm_fold nf = norm ? *norm : hm_norm_fold{nullptr, nullptr, 0.0f, 0};
    hipLaunchKernelGGL(router_partial_kernel, pgrid, dim3(HM_WAVE),
                       norm ? (size_t)hidden * sizeof(float) : 0, hm_stream(stream), h, w,
                       (int)hidden, (int)experts, part, fused ? fused->counters : nullptr,
                       fused ? fused->n_counters : 0, nf);
    HM_LAUNCHED();
    if (!select) return HM_OK;
    // the select kernel's fallback chains read the normalised rows
    if (norm) h = norm->x_out;
#define HM_SELECTP(N, F, W)                                                                \
    hipLaunchKernelGGL((router_select_partial_kernel<N, F, W, F>), sgrid, dim3(W * HM_WAVE), \
                       seq_bytes, hm_stream(stream), h, w, part, tokens, hidden, experts,    \
                       top_k, flags, logits, ids, scores, status,                            \
                       F ? fused->counters : nullptr, F ? fused->counts : nullptr,           \
                       F ? fused->offsets : nullptr, F ? fused->perm_tokens : nullptr,       \
                       F ? fused->perm_weights : nullptr, F ? fused->slots : nullptr, q)
#define HM_SELECTP2(N)                                  \
    do {                                                \
        if (!fused) HM_SELECTP(N, false, 4);            \
        else if (nw == 1) HM_SELECTP(N, true, 1);       \
        else if (nw == 2) HM_SELECTP(N, true, 2);       \
        else HM_SELECTP(N, true, 4);                    \
    } while (0)
    if (epl <= 1) HM_SELECTP2(1);
    else if (epl <= 2) HM_SELECTP2(2);
    else if (epl <= 4) HM_SELECTP2(4);
    else if (epl <= 8) HM_SELECTP2(8);
    else HM_SELECTP2(16);
#undef HM_SELECTP2
#undef HM_SELECTP
    HM_LAUNCHED();
    return HM_OK;
}

// One-token decode with the select inside the gate/up launch
// (select_gateup_kernel): the shapes it takes -- an INT8 layer whose
// gate/up the slice kernel covers (the token row in LDS, K tiles within four
// loads per wave), at most 8 rows of 64 logits, the partial kernel's H.
bool hm_select_gateup_ok(const hm_layer* L, int32_t top_k) {
    const int64_t KT = hm_pad32(L->hidden) / 32;
    // (E <= 128: the kernel's LDS holds two rows of block partials; H <= 2 x
    // 4 x 512 floats: the token row in two float4 per thread)
    return L->dtype == HM_DTYPE_INT8 && L->experts <= 2 * HM_WAVE && top_k >= 1 &&
           top_k <= L->experts && top_k <= kMaxTopK && L->hidden % kNB == 0 &&
           L->hidden <= 8 * kGvThreads && KT <= 16 * kGsQ && L->intermediate % 8 == 0;
}

// The first launch of such a step: the router partials (router_partial_kernel,
// which also zeroes the step's counters and, with `norm`, folds the RMSNorm
// in and writes norm->x_out).
int hm_route_partials_decode(const float* h, const float* w, int64_t hidden, int64_t experts,
                             int32_t top_k, uint32_t flags, int32_t* status, void* route_ws,
                             const hm_decode_fusion* fused, const hm_norm_fold* norm,
                             void* stream) {
    HM_REQUIRE(h && w && route_ws && fused && fused->counters && experts > 0 && hidden > 0);
    HM_REQUIRE(!norm || (norm->gamma && norm->x_out && std::isfinite(norm->eps) &&
                         norm->eps > 0.0f && hidden <= 16384));
    if (experts > 1024 || hidden % kNB != 0 || hidden > INT_MAX) return HM_ERR_UNSUPPORTED;
    return launch_decode_router(h, w, 1, hidden, experts, top_k, flags,
                                static_cast<float*>(route_ws), nullptr, nullptr, status, route_ws,
                                fused, norm, nullptr, stream, false);
}

// The second: select_gateup_kernel.  x: the token row the router read (the
// normalised one when the norm is folded); z [k x I]: SiLU(G) * U of the k
// selected experts' rows in ascending id; ids ... slots: the routing results
// and the groups (hm_route_permute_decode's).  The first kernel of the
// gate/up stage and its last (an armed stage timer brackets it).
int hm_launch_select_gateup(const float* x, const float* w, int32_t top_k, uint32_t flags,
                            uint32_t* ids, float* scores, int32_t* status, void* route_ws,
                            int32_t* counts, int32_t* offsets, int32_t* perm_tokens,
                            float* perm_weights, int32_t* slots, const hm_layer* L, float* z,
                            hipStream_t stream) {
    HM_REQUIRE(x && w && ids && scores && route_ws && counts && offsets && perm_tokens &&
               perm_weights && slots && z);
    if (!hm_select_gateup_ok(L, top_k)) return HM_ERR_UNSUPPORTED;
    const int64_t H = L->hidden, E = L->experts, I = L->intermediate;
    const int64_t KT = hm_pad32(H) / 32;
    float* logits = static_cast<float*>(route_ws);
    const double* part = reinterpret_cast<const double*>(static_cast<char*>(route_ws) +
                                                         route_logits_bytes(1, E));
    const dim3 grid((unsigned)(I / 8), (unsigned)top_k);
    const size_t lds = (size_t)H * sizeof(float);
    const int epl = (int)((E + HM_WAVE - 1) / HM_WAVE);
    const int lj = (int)((KT + kGsQ - 1) / kGsQ + 3) / 4;
#define HM_SG(EPL, LJ)                                                                          \
    HM_STAGE_LAUNCH(true, true, (select_gateup_kernel<EPL, LJ>), grid, dim3(kGvThreads), lds,   \
                    stream, x, w, part, H, E, top_k, flags, logits, ids, scores, status, counts, \
                    offsets, perm_tokens, perm_weights, slots, I,                                \
                    static_cast<const int8_t*>(L->packed), L->scale, L->zero_point, z)
#define HM_SG2(EPL)                                                                             \
    do {                                                                                        \
        if (lj <= 1) HM_SG(EPL, 1);                                                             \
        else if (lj <= 2) HM_SG(EPL, 2);                                                        \
        else HM_SG(EPL, 4);                                                                     \
    } while (0)
    if (epl <= 1) HM_SG2(1);
    else HM_SG2(2);
#undef HM_SG2
#undef HM_SG
    HM_LAUNCHED();
    return HM_OK;
}

// Routing and grouping of a decode batch (T <= 16) in two launches instead
// of hm_router_topk + hm_permute's three; same results.  Counter 0 of
// fused->counters is the select's completion counter; all n_counters are
// zeroed by the first launch.  With `norm`, h is the layer input and the
// router (and norm->x_out) get RMSNorm(h) (hm_rmsnorm's results).
int hm_route_permute_decode(const float* h, const float* w, int64_t tokens, int64_t hidden,
                            int64_t experts, int32_t top_k, uint32_t flags, uint32_t* ids,
                            float* scores, int32_t* status, void* route_ws,
                            const hm_decode_fusion* fused, const hm_norm_fold* norm,
                            const hm_row_quant* xq, bool* quantized, void* stream) {
    if (quantized) *quantized = false;
    HM_REQUIRE(experts > 0 && top_k > 0 && top_k <= experts && fused && fused->counters);
    HM_REQUIRE(h && w && ids && scores && route_ws && tokens > 0 && hidden > 0);
    // (the norm's row copy is hidden floats of LDS, as in hm_rmsnorm)
    HM_REQUIRE(!norm || (norm->gamma && norm->x_out && std::isfinite(norm->eps) &&
                         norm->eps > 0.0f && hidden <= 16384));
    if (experts > 1024 || top_k > kMaxTopK || tokens > kDecodeTokens || hidden % kNB != 0 ||
        tokens * top_k > kSmallPairs || hidden > INT_MAX)
        return HM_ERR_UNSUPPORTED;
    // the select kernel also cuts the rows' activation digits when asked
    // (widths the one-wave row quantisation takes; the rows it reads are the
    // normalised ones when the norm is folded in)
    const hm_row_quant* q =
        xq && xq->digits && xq->scales && xq->limbs >= 1 && xq->limbs <= 3 &&
                hidden % 256 == 0 && hidden / 256 <= kHmQuantMaxV &&
                (uintptr_t)xq->digits % 4 == 0 && (uintptr_t)(norm ? norm->x_out : h) % 16 == 0
            ? xq
            : nullptr;
    const int rc = launch_decode_router(h, w, tokens, hidden, experts, top_k, flags,
                                        static_cast<float*>(route_ws), ids, scores, status,
                                        route_ws, fused, norm, q, stream);
    if (rc == HM_OK && q && quantized) *quantized = true;
    return rc;
}

extern "C" {

__attribute__((visibility("hidden"))) int hm_router_topk_quant(const float* h, const float* w, int64_t tokens,
                         int64_t hidden, int64_t experts, int32_t top_k,
                         uint32_t flags, uint32_t* ids, float* scores,
                         float* logits_out, int32_t* status, void* route_ws,
                         const hm_row_quant* xq, bool* quantized, int32_t* hist,
                         bool* counted, void* stream);

__attribute__((visibility("hidden"))) int hm_permute_counted(const uint32_t* ids, const float* scores, int64_t tokens,
                       int32_t top_k, int64_t experts, int32_t* counts, int32_t* offsets,
                       int32_t* perm_tokens, float* perm_weights, int32_t* slots,
                       void* workspace, bool counted, void* stream);

int hm_router_topk(const float* h, const float* w, int64_t tokens,
                   int64_t hidden, int64_t experts, int32_t top_k,
                   uint32_t flags, uint32_t* ids, float* scores,
                   float* logits_out, int32_t* status, void* route_ws,
                   void* stream) {
    return hm_router_topk_quant(h, w, tokens, hidden, experts, top_k, flags, ids, scores,
                                logits_out, status, route_ws, nullptr, nullptr, nullptr,
                                nullptr, stream);
}

// hm_router_topk, and where a batch's select kernel runs, the rows of h
// quantised into xq's digit planes as well (*quantized tells the caller).
__attribute__((visibility("hidden"))) int hm_router_topk_quant(const float* h, const float* w, int64_t tokens,
                         int64_t hidden, int64_t experts, int32_t top_k,
                         uint32_t flags, uint32_t* ids, float* scores,
                         float* logits_out, int32_t* status, void* route_ws,
                         const hm_row_quant* xq, bool* quantized, int32_t* hist,
                         bool* counted, void* stream) {
    if (quantized) *quantized = false;
    if (counted) *counted = false;
    // RouterConfig::validate (src/router/RouterConfig.cpp:9-22)
    HM_REQUIRE(experts > 0 && top_k > 0 && top_k <= experts);
    HM_REQUIRE(h && w && ids && scores && tokens > 0 && hidden > 0);
    HM_REQUIRE(logits_out || route_ws);
    if (experts > 1024 || top_k > kMaxTopK) return HM_ERR_UNSUPPORTED;
    if (tokens > (int64_t)1 << 27) return HM_ERR_OVERFLOW;  // 32-bit grids
    float* logits = logits_out ? logits_out : static_cast<float*>(route_ws);
    const int epl = (int)((experts + HM_WAVE - 1) / HM_WAVE);
    const unsigned sel = (unsigned)((tokens + 3) / 4);
    const size_t seq_bytes = (size_t)(kBlock / HM_WAVE) * experts * sizeof(float);
    if (route_ws && tokens <= kDecodeTokens && hidden % kNB == 0 && hidden <= INT_MAX) {
        // decode: certified block partials, then select over the logits
        // formed from them
        return launch_decode_router(h, w, tokens, hidden, experts, top_k, flags, logits, ids,
                                    scores, status, route_ws, nullptr, nullptr, nullptr, stream);
    }
    hm_row_quant bq = {nullptr, nullptr, nullptr, 0};
    if (xq && xq->digits && xq->scales && xq->limbs >= 1 && xq->limbs <= 3 && hidden % 256 == 0 &&
        hidden / 256 <= kHmQuantMaxV && (uintptr_t)xq->digits % 4 == 0 && (uintptr_t)h % 16 == 0 &&
        tokens <= (int64_t)1 << 24)  // (twice the workgroups: 2^31 threads)
        bq = *xq;
    // the chunk histograms of hm_permute, when the caller passes them
    const int64_t chunks = (tokens * top_k + kPermChunk - 1) / kPermChunk;
    int32_t* hc = hist && chunks > 1 && chunks * experts <= INT_MAX ? hist : nullptr;
    const int hc_n = hc ? (int)(chunks * experts) : 0;
    if (quantized) *quantized = bq.digits != nullptr;
    if (counted) *counted = hc != nullptr;
    const int rc = launch_router_chains(h, w, tokens, hidden, experts, logits, status, hc, hc_n, stream);
    if (rc) return rc;
    const dim3 sgrid(bq.digits ? 2 * sel : sel);
#define HM_SELECT(N)                                                                   \
    hipLaunchKernelGGL(router_select_kernel<N>, sgrid, dim3(kBlock), seq_bytes,        \
                       hm_stream(stream), logits, tokens, experts, top_k, flags, ids,  \
                       scores, status, h, hidden, bq, hc, sel)
    if (epl <= 1) HM_SELECT(1);
    else if (epl <= 2) HM_SELECT(2);
    else if (epl <= 4) HM_SELECT(4);
    else if (epl <= 8) HM_SELECT(8);
    else HM_SELECT(16);
#undef HM_SELECT
    HM_LAUNCHED();
    return HM_OK;
}

// Permute workspace: the per-chunk histograms [chunks x E] (none for one
// chunk).
size_t hm_permute_workspace_bytes(int64_t tokens, int32_t top_k, int64_t experts) {
    if (tokens <= 0 || top_k <= 0 || experts <= 0) return 0;
    const int64_t chunks = (tokens * top_k + kPermThreads - 1) / kPermThreads;
    return chunks > 1 ? (size_t)chunks * (size_t)experts * sizeof(int32_t) : 0;
}

int hm_permute(const uint32_t* ids, const float* scores, int64_t tokens,
               int32_t top_k, int64_t experts, int32_t* counts, int32_t* offsets,
               int32_t* perm_tokens, float* perm_weights, int32_t* slots,
               void* workspace, void* stream) {
    return hm_permute_counted(ids, scores, tokens, top_k, experts, counts, offsets,
                              perm_tokens, perm_weights, slots, workspace, false, stream);
}

// hm_permute; `counted`: the workspace already holds the chunk histograms
// (the prefill router's select kernel counted them), so only the scatter runs.
__attribute__((visibility("hidden"))) int hm_permute_counted(const uint32_t* ids, const float* scores, int64_t tokens,
                       int32_t top_k, int64_t experts, int32_t* counts, int32_t* offsets,
                       int32_t* perm_tokens, float* perm_weights, int32_t* slots,
                       void* workspace, bool counted, void* stream) {
    HM_REQUIRE(ids && scores && counts && offsets && perm_tokens && perm_weights && slots);
    HM_REQUIRE(tokens > 0 && top_k > 0 && experts > 0 && top_k <= experts);
    if (experts > 1024) return HM_ERR_UNSUPPORTED;
    if (tokens * top_k > INT_MAX) return HM_ERR_OVERFLOW;
    const int64_t pairs = tokens * top_k;
    const int64_t chunks = (pairs + kPermThreads - 1) / kPermThreads;
    int32_t* hist = nullptr;
    if (chunks > 1) {
        HM_REQUIRE(workspace);
        hist = static_cast<int32_t*>(workspace);
    }
    if (chunks > 1 && !counted) {
        hipLaunchKernelGGL(permute_count_kernel, dim3((unsigned)chunks), dim3(kPermThreads), 0,
                           hm_stream(stream), ids, pairs, experts, hist);
        HM_LAUNCHED();
    }
    hipLaunchKernelGGL(permute_scatter_kernel, dim3((unsigned)chunks), dim3(kPermThreads), 0,
                       hm_stream(stream), ids, scores, pairs, top_k, experts, hist, chunks,
                       counts, offsets, perm_tokens, perm_weights, slots);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_gather_rows(const float* in, const int32_t* rows, int64_t count,
                   int64_t width, float* out, void* stream) {
    HM_REQUIRE(in && rows && out && count >= 0 && width > 0);
    if (count == 0) return HM_OK;
    HM_REQUIRE(count <= 65535);
    const unsigned gx = (unsigned)((width + kBlock - 1) / kBlock > 64 ? 64 : (width + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(gather_rows_kernel, dim3(gx, (unsigned)count), dim3(kBlock), 0,
                       hm_stream(stream), in, rows, count, width, out);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_combine(const float* y_grouped, const uint32_t* ids, const int32_t* slots,
               const float* scores, int64_t tokens, int32_t top_k, int64_t width,
               const float* residual, float* out, void* stream) {
    HM_REQUIRE(y_grouped && ids && slots && scores && out);
    HM_REQUIRE(tokens > 0 && top_k > 0 && width > 0);
    if (top_k > kMaxTopK) return HM_ERR_UNSUPPORTED;
    HM_REQUIRE(tokens <= INT_MAX);
    hipLaunchKernelGGL(combine_kernel, dim3((unsigned)tokens), dim3(kBlock), 0,
                       hm_stream(stream), y_grouped, ids, slots, scores, tokens, top_k,
                       width, residual, out);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_silu(const float* x, float* y, int64_t n, void* stream) {
    HM_REQUIRE(x && y && n >= 0);
    if (n == 0) return HM_OK;
    hipLaunchKernelGGL(silu_kernel, dim3(grid_for(n)), dim3(kBlock), 0, hm_stream(stream), x, y, n);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_mul(const float* a, const float* b, float* y, int64_t n, void* stream) {
    HM_REQUIRE(a && b && y && n >= 0);
    if (n == 0) return HM_OK;
    hipLaunchKernelGGL(mul_kernel, dim3(grid_for(n)), dim3(kBlock), 0, hm_stream(stream), a, b, y, n);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_add(const float* a, const float* b, float* y, int64_t n, void* stream) {
    HM_REQUIRE(a && b && y && n >= 0);
    if (n == 0) return HM_OK;
    hipLaunchKernelGGL(add_kernel, dim3(grid_for(n)), dim3(kBlock), 0, hm_stream(stream), a, b, y, n);
    HM_LAUNCHED();
    return HM_OK;
}

int hm_debug_expf(const float* x, float* y, int64_t n, void* stream) {
    HM_REQUIRE(x && y && n >= 0);
    if (n == 0) return HM_OK;
    hipLaunchKernelGGL(expf_kernel, dim3(grid_for(n)), dim3(kBlock), 0, hm_stream(stream), x, y, n);
    HM_LAUNCHED();
    return HM_OK;
}

}  // extern "C"
