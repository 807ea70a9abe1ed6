// Fragment-ordered projections for the denoise loop's few rows (gfx950).
//
// Replaces, for the block projections of a model step, gemm_bias_act (src/backend/cuda/cuda_backend.cu:337-467)
// with the ops around it -- split_qkv + apply_qk_norm, the residual add and
// the RMSNorm that follows (dit_block.cu:198-387) -- by ONE launch per
// projection.
//
// Fragment order.  A matrix X[R][K] of 16-bit elements is stored as 1 KB
// blocks of 16 rows x 32 columns, block (r / 16, k / 32) at index
// (r / 16) * (K / 32) + k / 32, and inside a block lane l = 16 ((k % 32) / 8)
// + r % 16 of a wave holds the 8 elements k % 8: exactly the operand of one
// v_mfma_f32_16x16x32.  int8 codes: blocks of 16 rows x 64 columns, lane l
// holds the 8 codes of step 64 kc + 8 (l / 16) .. + 7 and the 8 of the step
// 32 columns further.  So an operand load of a wave is 1 KB of contiguous
// memory.  Read from row-major rows the same operand is 16 pieces of 64
// bytes, and each piece costs the address path what a whole 128-byte line
// does: the same kernel over the same bytes took 9.7 us row-major and
// 5.9 us in fragment order (67 x 2048 x 2048, cold weights, graph-timed).
//
// At that rate one workgroup can afford all of K, so there are no K-slice
// partials to write, flush and read back and no reduce launch.  Graph-timed on
// cold weights, 67 rows: 2048 x 2048 6.0-6.2 us with any epilogue against 7.3
// for split-K + the plain reduce, 8.5 for its deferred and 10.0 for its
// row-wide residual add + RMSNorm; the 6144 x 2048 QKV projection 10.7 against
// 14.3.  The batch-1 loop went from 11.3 to 9.4 ms.  An empty launch takes
// 1.65 us, the weights 1.5 us at the rate a large read reaches; with everything
// in L2 the 2048 x 2048 call takes 4.4 us.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "sf_act.h"
#include "sf_device.h"
#include "sf_hip.h"

namespace sfk {

constexpr int kFragWaves = 4;
constexpr size_t kFragLds = 160 * 1024;
constexpr int kFragRowTiles = 64;   // tile sums of a deferred row: 16 in each of 4 lane groups

// What the rows of a are (the RS template argument): finished; x * gamma of a
// deferred norm in bf16; or that in fp16 with the range guard.
//
// The guard.  x * gamma, unlike the normalised row, is neither bounded by
// fp16's range nor kept out of its subnormals.  The producer of the row marks
// both in the tile sums that the consumer reads anyway: an element beyond the
// range by an infinite sum, and a tile without an element of at least
// sqrt(N) 2^-11 by a negative one.  A row is contracted again from the fp32
// residual, normalised first, by the wave that finishes it, if its sum is
// infinite, or if all its tiles are negative and its mean square is below 1.
// Any other row is stored no worse than a normalised one: with an element of
// sqrt(N) 2^-11 its rms is at least 2^-11, of which the half step of a
// subnormal, 2^-25, is an eighth of the error that an 11-bit rounding may make;
// with a mean square of at least 1 each x * gamma is at least as large as the
// normalised element.  Rows in range, every row of a model whose residual is
// not degenerate, pay the comparison; a row's result does not depend on whether
// its neighbours are in range.  A row that falls back takes its workgroup through
// K again with scalar loads: 67 x 2048 x 2048 takes 30 us against 5.6 with one
// such row or all of them, 402 x 6144 112 us with one and 309 with all against 22.
enum RowKind { kRowPlain = 0, kRowDeferred = 1, kRowGuarded = 2 };
constexpr float kF16Max = 65504.f;
inline float guard_min(int cols) { return sqrtf((float)cols) / 2048.f; }   // the mark of a row of cols

// The epilogue's arguments (the operands' pointers and sizes are scalar kernel
// arguments of their own, see gemm_frag_kernel).
struct FragEpi {
    const float* bias;     // [N] or null
    const float* w_scale;  // [N] (int8 weights)
    int N;
    int act;
    int c_kind;            // plain: 0 fp32, 1 bf16, 2 fp16
    int c_frag;            // plain: fragment order (16-bit), else row-major [M][ldc]
    int accumulate;        // plain: fp32 c += result
    void* c;               // plain output; the residual of the add + norm
    int64_t ldc;
    // residual add + deferred RMSNorm: c (fp32) += result; norm_out (fragment
    // order) = c * gamma; norm_ss[m][tile] = the tile's sum of c^2
    const float* norm_gamma;
    uint16_t* norm_out;
    float* norm_ss;
    float norm_min;   // fp16: the range guard's mark (guard_min); bf16: 0
    // kRowGuarded: the fp32 rows [M][x_ld] and the norm's gamma
    const float* x;
    const float* x_gamma;
    int64_t x_ld;
    // per-head
    int H, S;
    float eps;
    const float* head_gamma[3];
    uint16_t* head_out[3];
    int64_t head_sb[3], head_sh[3], head_ss[3];
};

__device__ __forceinline__ uint2 pack_kind4(f32x4 v, bool f16) {
    return f16 ? uint2{pack_f16x2_rn(v[0], v[1]), pack_f16x2_rn(v[2], v[3])}
               : uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// Sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 that share an MFMA column.
__device__ __forceinline__ float sum_groups(float x) {
    auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// Whether x holds in any of those four lanes (a few scalar operations on the
// comparison's mask: the epilogue that asks is the end of its wave's path).
__device__ __forceinline__ bool any_groups(bool x) {
    uint64_t q = __ballot(x);
    q |= q >> 32;
    q |= q >> 16;
    return __builtin_amdgcn_inverse_ballot_w64((q & 0xffff) * 0x0001000100010001ull);
}

// One workgroup of 4 waves per (16 NB columns x 16 MB rows) of C over all of
// K: wave w contracts its quarter of K with both operands loaded straight into
// registers -- nothing is shared between waves, so nothing is staged and no
// wave waits for another -- NG groups of U units in flight (a unit is one
// 32-wide MFMA step, two for int8), and the four waves' fp32 accumulators meet
// in LDS, RB row blocks at a time.  C^T = W . A^T, so weight rows are MFMA
// rows: accumulator [nb][mb] holds column 16 nb + 4 g + i and row 16 mb + r in
// lane 16 g + r.  The waves then finish items of one row block x EN column
// blocks: the four sums in wave order, scale, the deferred norm's row scale,
// bias, activation and the epilogue.
//
// What bounds it: a CU moves 64 bytes a clock through its address path and
// cache, so (NB + MB) KB per step and wave, and the tile is chosen for few
// bytes per CU (frag_tile); the row splits of a column tile run on one XCD
// (workgroup ids congruent mod 8), whose L2 then serves the weights to all but
// the first.  The accumulators are the price of not staging: 4 NB MB registers
// of the 512 a wave has to itself.
//
// The operands' pointers and the sizes are separate scalar arguments at the
// front: those are preloaded into SGPRs with the wave
// (-amdgpu-kernarg-preload-count), so the first loads go out without a
// scalar-memory round trip; the epilogue's arguments are fetched behind them.
template <int NB, int MB, int U, int NG, bool W8, bool AH, int EPI, int RS>
__global__ __launch_bounds__(64 * kFragWaves) __attribute__((amdgpu_waves_per_eu(1, 2))) void gemm_frag_kernel(
    const void* A, const void* W, int K, int M, int ntiles, const float* row_ss, int row_tiles, float row_inv_n,
    float row_eps, const FragEpi e) {
    static_assert(EPI != SF_EPI_HEADS || NB == 4, "a head is one column tile");
    static_assert(RS == kRowPlain || (AH ? RS == kRowGuarded && EPI == SF_EPI_PLAIN : RS == kRowDeferred),
                  "deferred fp16 rows are guarded, and taken by the plain epilogue only");
    constexpr int NW = kFragWaves;
    constexpr int ST = W8 ? 2 : 1;         // MFMA steps per unit: 16 bytes of codes are two steps
    constexpr bool kAddNorm = EPI == SF_EPI_ADD_NORM, kHeads = EPI == SF_EPI_HEADS, kPlain = EPI == SF_EPI_PLAIN;
    constexpr int EN = NB < 4 ? NB : 4;    // column blocks of an item
    constexpr int IT = NB / EN;            // items per row block
    constexpr int RB = (size_t)NW * NB * MB * 1024 <= kFragLds ? MB : (MB + 1) / 2;   // row blocks in LDS at once
    static_assert((size_t)NW * NB * RB * 1024 <= kFragLds && NW % IT == 0, "accumulators in LDS, a wave's items in one column half");
    constexpr int NI = (RB * IT + NW - 1) / NW;   // items of a wave per round of RB row blocks
    // Where the registers allow, the items' operands are fetched ahead of the
    // contraction, else behind its last loads.
    constexpr bool kEarly = NB * MB <= 20;
    __shared__ __attribute__((aligned(16))) f32x4 red[NW * NB * RB * 64];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int g4 = lane >> 4, r = lane & 15;
    const int ms = (int)blockIdx.x >> 3;
    const int tile = ((int)blockIdx.x & 7) + 8 * (int)blockIdx.y;
    if (tile >= ntiles) return;   // the last group of 8 tiles is padded
    const int n0 = tile * 16 * NB, m0 = ms * 16 * MB;
    const int rows16 = min((M + 15) / 16 - ms * MB, MB) * 16;   // stored rows of this tile
    const __amdgpu_buffer_rsrc_t ars =
        make_rsrc(static_cast<const char*>(A) + (int64_t)m0 * K * 2, (uint32_t)(rows16 * K * 2));
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(static_cast<const char*>(W) + (int64_t)n0 * K * (W8 ? 1 : 2),
                                                 (uint32_t)(16 * NB * K * (W8 ? 1 : 2)));
    const int steps = K >> 5;
    const int nu = steps / ST;                                      // units
    const int per = (2 / ST) * (((K >> 6) + NW - 1) / NW);          // a wave's share: whole 64-wide chunks
    const int cb = w * per, ce = min(nu, cb + per);

    // RS: the rows' tile sums, row-major so that lane group g4 fetches tiles
    // 16 q + 4 g4 .. + 3 of row r as 16 bytes (q < 4).
    auto load_row = [&](int m, f32x4 (&v)[kFragRowTiles / 16]) {
        const __amdgpu_buffer_rsrc_t rrs = make_rsrc(row_ss, (uint32_t)(row_tiles * M * 4));
#pragma unroll
        for (int q = 0; q < kFragRowTiles / 16; ++q) {
            const int t = 16 * q + 4 * g4;
            const uint32_t off = (uint32_t)((m * row_tiles + t) * 4) | ((m < M) & (t < row_tiles) ? 0u : 0x80000000u);
            v[q] = __builtin_bit_cast(f32x4, buffer_load16(rrs, off));
        }
    };
    auto row_sum = [&](f32x4 (&v)[kFragRowTiles / 16], bool& marked) {
        if (row_tiles & 3) {   // the last quad runs into the next row
#pragma unroll
            for (int q = 0; q < kFragRowTiles / 16; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[q][i] = 16 * q + 4 * g4 + i < row_tiles ? v[q][i] : 0.f;
        }
        if constexpr (RS == kRowGuarded) {   // marked: every tile's sum is negative (or zero)
            float top = 0.f;
#pragma unroll
            for (int q = 0; q < kFragRowTiles / 16; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    top = fmaxf(top, v[q][i]);
                    v[q][i] = fabsf(v[q][i]);
                }
            marked = !any_groups(top > 0.f);
        }
        const f32x4 t = (v[0] + v[1]) + (v[2] + v[3]);
        return sum_groups((t[0] + t[1]) + (t[2] + t[3]));
    };
    // Items of wave w in the round of row blocks p0 .. p0 + RB - 1: row block
    // p0 + (w + 4 k) / IT, k < NI, and always the column half it = w % IT.
    const int it = w % IT;
    auto item_mb = [&](int p0, int k) { return (w + NW * k) < RB * IT ? p0 + (w + NW * k) / IT : MB; };
    f32x4 bias[EN], scale[EN], gam[EN];   // of the wave's columns
    f32x4 res[NI][EN], rss[NI][kFragRowTiles / 16];   // residual and tile sums of the items' rows
    auto load_cols = [&] {
        const __amdgpu_buffer_rsrc_t brs = make_rsrc(e.bias, e.bias ? (uint32_t)(e.N * 4) : 0u);   // null: zeros
        const __amdgpu_buffer_rsrc_t srs = make_rsrc(e.w_scale, W8 ? (uint32_t)(e.N * 4) : 0u);
        const __amdgpu_buffer_rsrc_t grs = make_rsrc(e.norm_gamma, kAddNorm ? (uint32_t)(e.N * 4) : 0u);
#pragma unroll
        for (int j = 0; j < EN; ++j) {
            const uint32_t n = (uint32_t)(n0 + 16 * (EN * it + j) + 4 * g4);
            bias[j] = __builtin_bit_cast(f32x4, buffer_load16(brs, n * 4));
            scale[j] = W8 ? __builtin_bit_cast(f32x4, buffer_load16(srs, n * 4)) : f32x4{1.f, 1.f, 1.f, 1.f};
            if constexpr (kAddNorm) gam[j] = __builtin_bit_cast(f32x4, buffer_load16(grs, n * 4));
        }
    };
    auto load_rows = [&](int p0) {   // rows past M, and items past MB, read as zeros
        if constexpr (kAddNorm || kPlain) {
            const bool need_res = kAddNorm || e.accumulate;
            const __amdgpu_buffer_rsrc_t xrs =
                make_rsrc(static_cast<const char*>(e.c) + (need_res ? (int64_t)m0 * e.ldc * 4 : 0),
                          need_res ? (uint32_t)(min(16 * MB, M - m0) * e.ldc * 4) : 0u);
#pragma unroll
            for (int k = 0; k < NI; ++k)
#pragma unroll
                for (int j = 0; j < EN; ++j)
                    res[k][j] = __builtin_bit_cast(
                        f32x4, buffer_load16(xrs, (uint32_t)(((16 * item_mb(p0, k) + r) * e.ldc + n0 + 16 * (EN * it + j) + 4 * g4) * 4)));
        }
    };
    auto load_sums = [&](int p0) {
#pragma unroll
        for (int k = 0; k < NI; ++k) load_row(item_mb(p0, k) < MB ? m0 + 16 * item_mb(p0, k) + r : M, rss[k]);
    };
    float sum[NI], rs[NI];
    bool marked[NI];
    auto row_scales = [&] {
#pragma unroll
        for (int k = 0; k < NI; ++k) {
            sum[k] = row_sum(rss[k], marked[k]);
            rs[k] = deferred_rsqrt(sum[k], row_inv_n, row_eps);
        }
    };
    // ahead of the operands, so the row scales are formed while those are under way
    if constexpr (RS != kRowPlain && kEarly) load_sums(0);
    __builtin_amdgcn_sched_barrier(0);

    constexpr int UP = U % 2 ? 1 : 2;
    u32x4 wv[NG][U][NB], av[NG][U][ST * MB];
    // One group of U units; units past ce load zeros (beyond the buffer
    // range, no traffic).  Two neighbouring units are 2 KB of a row block.
    // Always issued, so that the count of loads in
    // flight is known and each wait covers one operand at a time.
    auto issue_w = [&](int c0, u32x4 (&ww)[U][NB]) {
#pragma unroll
        for (int t = 0; t < U; t += UP)
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int p = t; p < t + UP; ++p) {
                    const uint32_t off = (uint32_t)(lane * 16) | (c0 + p < ce ? 0u : 0x80000000u);
                    ww[p][i] = __builtin_amdgcn_raw_buffer_load_b128(wrs, off, (i * nu + (c0 + p < ce ? c0 + p : 0)) * 1024, 0);
                }
    };
    auto issue_a = [&](int c0, u32x4 (&aa)[U][ST * MB]) {
#pragma unroll
        for (int t = 0; t < U; t += UP)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int p = t; p < t + UP; ++p)
#pragma unroll
                    for (int s = 0; s < ST; ++s) {
                        const uint32_t off = (uint32_t)(lane * 16) | (c0 + p < ce ? 0u : 0x80000000u);
                        aa[p][ST * i + s] = __builtin_amdgcn_raw_buffer_load_b128(
                            ars, off, (i * steps + ST * (c0 + p < ce ? c0 + p : 0) + s) * 1024, 0);
                    }
    };
    f32x4 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mm = [&](const u32x4 (&ww)[U][NB], const u32x4 (&aa)[U][ST * MB]) {
#pragma unroll
        for (int t = 0; t < U; ++t)
#pragma unroll
            for (int s = 0; s < ST; ++s) {
                u32x4 wf[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    if constexpr (W8) {
                        const uint2 q = {ww[t][nb][2 * s], ww[t][nb][2 * s + 1]};
                        if constexpr (AH) wf[nb] = __builtin_bit_cast(u32x4, i8x8_to_f16x8(q));
                        else wf[nb] = __builtin_bit_cast(u32x4, i8x8_to_bf16x8(q));
                    } else {
                        wf[nb] = ww[t][nb];
                    }
                }
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        if constexpr (AH)
                            acc[nb][mb] = mfma16x16x32_f16(u32x4_as_f16x8(wf[nb]), u32x4_as_f16x8(aa[t][ST * mb + s]), acc[nb][mb]);
                        else
                            acc[nb][mb] = mfma16x16x32(u32x4_as_bf16x8(wf[nb]), u32x4_as_bf16x8(aa[t][ST * mb + s]), acc[nb][mb]);
                    }
            }
    };
    // Weights first: they come from HBM; the epilogue's operands and the
    // activations, from the L2 or the memory-side cache, while the weights
    // are under way.  (The barriers: the compiler would sink the loads next
    // to their uses.)
#pragma unroll
    for (int b = 0; b < NG; ++b) issue_w(cb + b * U, wv[b]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kEarly) {
        load_cols();
        load_rows(0);
    }
#pragma unroll
    for (int b = 0; b < NG; ++b) issue_a(cb + b * U, av[b]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (RS != kRowPlain && kEarly) row_scales();

    int c0 = cb;
    for (; c0 + NG * U < ce; c0 += NG * U) {
#pragma unroll
        for (int b = 0; b < NG; ++b) {
            mm(wv[b], av[b]);
            __builtin_amdgcn_sched_barrier(0);
            issue_w(c0 + (NG + b) * U, wv[b]);
            issue_a(c0 + (NG + b) * U, av[b]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int b = 0; b < NG; ++b) {
        if (b < 2 || c0 + b * U < ce) mm(wv[b], av[b]);   // groups past ce are zeros
        if (b == 0 && !kEarly) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (RS != kRowPlain) load_sums(0);
            load_cols();
            load_rows(0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

#pragma unroll
    for (int p0 = 0; p0 < MB; p0 += RB) {
    if (p0) {
        if constexpr (RS != kRowPlain) load_sums(p0);
        load_rows(p0);
        __syncthreads();   // the previous row blocks are finished
    }
#pragma unroll
    for (int mb = 0; mb < RB; ++mb)
        if (p0 + mb < MB) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) red[((w * RB + mb) * NB + nb) * 64 + lane] = acc[nb][p0 + mb < MB ? p0 + mb : 0];
        }
    __syncthreads();
    if constexpr (RS != kRowPlain) {
        if (!kEarly || p0) row_scales();
    }
    if (!W8 && e.w_scale) {   // 16-bit copies of int8 codes
#pragma unroll
        for (int j = 0; j < EN; ++j) scale[j] = *reinterpret_cast<const f32x4*>(e.w_scale + n0 + 16 * (EN * it + j) + 4 * g4);
    }
#pragma unroll
    for (int k = 0; k < NI; ++k) {
        const int mb = item_mb(p0, k);
        if (mb >= MB) continue;
        const int m = m0 + 16 * mb + r;
        f32x4 v[EN];
#pragma unroll
        for (int j = 0; j < EN; ++j) {
            v[j] = red[((mb - p0) * NB + EN * it + j) * 64 + lane];
#pragma unroll
            for (int s = 1; s < NW; ++s) v[j] += red[((s * RB + mb - p0) * NB + EN * it + j) * 64 + lane];
        }
        if constexpr (RS == kRowGuarded) {
            const float mean = sum[k] * row_inv_n;
            const bool out = m < M && !(mean < INFINITY && (mean >= 1.f || !marked[k]));
            if (__any(out)) {   // lanes r, r + 16, r + 32, r + 48 agree
                const float* xr = e.x + (int64_t)min(m, M - 1) * e.x_ld;
                float t = 0.f;
                for (int c = 8 * g4; c < K; c += 32)
#pragma unroll
                    for (int j = 0; j < 8; ++j) t += xr[c + j] * xr[c + j];
                const float inv_rms = 1.f / sqrtf(sum_groups(t) / (float)K + row_eps);
                f32x4 z[EN];
#pragma unroll
                for (int j = 0; j < EN; ++j) z[j] = f32x4{0.f, 0.f, 0.f, 0.f};
                for (int c = 0; c < steps; ++c) {
                    const int d = 32 * c + 8 * g4;
                    f16x8 f;
#pragma unroll
                    for (int j = 0; j < 8; ++j) f[j] = (_Float16)(xr[d + j] * inv_rms * e.x_gamma[d + j]);
#pragma unroll
                    for (int j = 0; j < EN; ++j) {
                        const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(wrs, (uint32_t)(lane * 16),
                                                                              ((EN * it + j) * nu + c / ST) * 1024, 0);
                        f16x8 wf;
                        if constexpr (W8) wf = i8x8_to_f16x8(c & 1 ? uint2{q[2], q[3]} : uint2{q[0], q[1]});
                        else wf = u32x4_as_f16x8(q);
                        z[j] = mfma16x16x32_f16(wf, f, z[j]);
                    }
                }
                if (out) {
                    rs[k] = 1.f;
#pragma unroll
                    for (int j = 0; j < EN; ++j) v[j] = z[j];
                }
            }
        }
        if constexpr (RS != kRowPlain) {
#pragma unroll
            for (int j = 0; j < EN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) v[j][q] = deferred_affine(v[j][q], scale[j][q], rs[k], bias[j][q]);
        } else {
#pragma unroll
            for (int j = 0; j < EN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) v[j][q] = v[j][q] * scale[j][q] + bias[j][q];
        }
        if constexpr (kHeads) {
            const int cols = e.H * 64;
            const int sec = n0 / cols, h = (n0 % cols) / 64;
            const float* gamma = e.head_gamma[sec];
            if (gamma) {   // rms_norm_kernel_impl over the 64 head dims (norm.cuh:89-122)
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < EN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) ss += v[j][q] * v[j][q];
                const float inv_rms = 1.f / sqrtf(sum_groups(ss) / 64.f + e.eps);
#pragma unroll
                for (int j = 0; j < EN; ++j) {
                    const f32x4 gq = *reinterpret_cast<const f32x4*>(gamma + 16 * j + 4 * g4);
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[j][q] = v[j][q] * inv_rms * gq[q];
                }
            }
            if (m >= M) continue;
            uint16_t* o = e.head_out[sec] + (int64_t)(m / e.S) * e.head_sb[sec] + h * e.head_sh[sec] +
                          (int64_t)(m % e.S) * e.head_ss[sec];
#pragma unroll
            for (int j = 0; j < EN; ++j) *reinterpret_cast<uint2*>(o + 16 * j + 4 * g4) = pack_kind4(v[j], false);
        } else if constexpr (kAddNorm) {
            const bool norm_f16 = e.norm_min > 0.f;
            float ss = 0.f, top = 0.f;
            f32x4 u[EN];
#pragma unroll
            for (int j = 0; j < EN; ++j) {
                v[j] += res[k][j];
                u[j] = v[j] * gam[j];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    ss += v[j][q] * v[j][q];
                    top = fmaxf(top, fabsf(u[j][q]));
                }
            }
            if (norm_f16 && top > kF16Max) ss = INFINITY;   // the guard's marks
            ss = sum_groups(ss);
            if (!any_groups(top >= e.norm_min)) ss = -ss;
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < EN; ++j) {
                const int n = n0 + 16 * (EN * it + j) + 4 * g4;
                *reinterpret_cast<f32x4*>(static_cast<float*>(e.c) + (int64_t)m * e.ldc + n) = v[j];
                *reinterpret_cast<uint2*>(e.norm_out + frag_off(m, n, e.N)) = pack_kind4(u[j], norm_f16);
            }
            if (g4 == 0) e.norm_ss[(int64_t)m * (ntiles * IT) + tile * IT + it] = ss;
        } else {
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < EN; ++j) {
                const int n = n0 + 16 * (EN * it + j) + 4 * g4;
#pragma unroll
                for (int q = 0; q < 4; ++q) v[j][q] = apply_act(e.act, v[j][q]);
                if (e.c_frag) {
                    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(e.c) + frag_off(m, n, e.N)) = pack_kind4(v[j], e.c_kind == 2);
                } else if (e.c_kind == 0) {
                    *reinterpret_cast<f32x4*>(static_cast<float*>(e.c) + (int64_t)m * e.ldc + n) =
                        e.accumulate ? res[k][j] + v[j] : v[j];
                } else {
                    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(e.c) + (int64_t)m * e.ldc + n) = pack_kind4(v[j], e.c_kind == 2);
                }
            }
        }
    }
    }
}

// RMSNorm of fp32 rows into fragment order, one workgroup of 256 threads per
// row (rms_norm_kernel_impl, norm.cuh:89-122).  Thread t owns columns
// 8 t .. 8 t + 7 (and 2048 further), one 16-byte store each.  ss != null: the
// deferred form instead -- x * gamma, and ss[row][t] = the sum of x^2 over the
// 64 columns of tile t.
constexpr int kNormFragPer = 2;   // cols <= 2 * 256 * 8 = 4096
__global__ __launch_bounds__(256) void norm_frag_kernel(const float* x, int64_t ldx, const float* gamma, uint16_t* out,
                                                        int f16, float* ss, int cols, float eps, float min_top) {
    __shared__ float red[4];
    const int row = blockIdx.x;
    f32x4 v[kNormFragPer][2], gq[kNormFragPer][2];
    float sum[kNormFragPer];
#pragma unroll
    for (int i = 0; i < kNormFragPer; ++i) {
        const int c = 8 * ((int)threadIdx.x + 256 * i);
        sum[i] = 0.f;
        if (c < cols) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v[i][h] = *reinterpret_cast<const f32x4*>(x + row * ldx + c + 4 * h);
                gq[i][h] = *reinterpret_cast<const f32x4*>(gamma + c + 4 * h);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j) sum[i] += v[i][h][j] * v[i][h][j];
        }
    }
    float s = 1.f;
    if (ss) {   // 8 lanes hold a 64-column tile
#pragma unroll
        for (int i = 0; i < kNormFragPer; ++i) {
            bool small = false;
            if (f16) {   // as the add + norm epilogue marks it
                float top = 0.f;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < 4; ++j) top = fmaxf(top, fabsf(v[i][h][j] * gq[i][h][j]));
                if (top > kF16Max) sum[i] = INFINITY;
                small = !((__ballot(top >= min_top) >> (threadIdx.x & 56)) & 255);
            }
            const float t = row8_sum(sum[i]) * (small ? -1.f : 1.f);
            const int c = 8 * ((int)threadIdx.x + 256 * i);
            if (c < cols && (threadIdx.x & 7) == 0) ss[(int64_t)row * (cols / 64) + c / 64] = t;
        }
    } else {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < kNormFragPer; ++i) t += sum[i];
        t = sum_groups(row16_sum(t));
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
        __syncthreads();
        s = 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)cols + eps);
    }
#pragma unroll
    for (int i = 0; i < kNormFragPer; ++i) {
        const int c = 8 * ((int)threadIdx.x + 256 * i);
        if (c < cols) {
            const uint2 lo = pack_kind4(v[i][0] * s * gq[i][0], f16 != 0);
            const uint2 hi = pack_kind4(v[i][1] * s * gq[i][1], f16 != 0);
            *reinterpret_cast<u32x4*>(out + frag_off(row, c, cols)) = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
    }
}

// Weight copies in fragment order: 16 bytes of the copy per thread, bf16 kept
// or rounded to the nearest fp16 (as sf_weights_to_f16 rounds), int8 codes
// kept or widened to fp16 (exact).  The reads of 16 rows x 64 bytes are gathered by one wave.
struct FragJobs {
    const void* w[SF_CODES_MAX_JOBS];
    void* out[SF_CODES_MAX_JOBS];
    int64_t ldw[SF_CODES_MAX_JOBS];
    int32_t K[SF_CODES_MAX_JOBS];
    int32_t kind[SF_CODES_MAX_JOBS];   // 0 copy 16-bit, 1 bf16 -> fp16, 2 int8, 3 int8 -> fp16
    uint32_t start[SF_CODES_MAX_JOBS + 1];
    int32_t count;
};

__global__ __launch_bounds__(256) void frag_pack_kernel(const FragJobs J) {
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= J.start[J.count]) return;
    int j = 0;
#pragma unroll
    for (int i = 1; i < SF_CODES_MAX_JOBS; ++i)
        if (i < J.count && idx >= J.start[i]) j = i;
    const uint32_t local = idx - J.start[j];
    const uint32_t lane = local & 63u, blk = local >> 6;
    const bool i8 = J.kind[j] == 2;
    const uint32_t kc = (uint32_t)J.K[j] / (i8 ? 64u : 32u);
    const uint32_t rb = blk / kc, c = blk - rb * kc;
    const int64_t row = 16 * (int64_t)rb + (lane & 15u);
    const uint32_t g4 = lane >> 4;
    u32x4 o;
    if (i8) {
        const int8_t* src = static_cast<const int8_t*>(J.w[j]) + row * J.ldw[j] + 64u * c + 8u * g4;
        const uint2 lo = *reinterpret_cast<const uint2*>(src), hi = *reinterpret_cast<const uint2*>(src + 32);
        o = u32x4{lo.x, lo.y, hi.x, hi.y};
    } else if (J.kind[j] == 3) {
        o = __builtin_bit_cast(
            u32x4, i8x8_to_f16x8(*reinterpret_cast<const uint2*>(static_cast<const int8_t*>(J.w[j]) + row * J.ldw[j] + 32u * c + 8u * g4)));
    } else {
        o = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(J.w[j]) + row * J.ldw[j] + 32u * c + 8u * g4);
        if (J.kind[j] == 1) o = __builtin_bit_cast(u32x4, bf16x8_to_f16x8(o));
    }
    *(static_cast<u32x4*>(J.out[j]) + local) = o;
}

// Tile of a call: NB 16-column blocks x MB 16-row blocks.  A CU runs one
// workgroup at a time and its time follows the operand bytes it fetches,
// (NB + MB) * 32 K, so the smallest rounds-of-256-workgroups * (NB + MB) is
// taken, on a tie the narrower one.  Graph-timed, cold weights, K = 2048, the
// kernel with a plain fp16 epilogue: 67 x 2048 (2, 2) 6.0 us against 7.0 for
// (2, 3) and 8.5 for (4, 2); 134 x 2048 (2, 3) 7.4 against 9.7 for (2, 2); 402 x
// 2048 (4, 4) 10.2 against 11.4 for (4, 5); 1072 x 2048 (8, 5) 16.5 against
// 22.1 for (4, 5) and 17.8 for (8, 6); 67 x 6144 (4, 3) 11.3 against 14.2 for
// (4, 2); 1072 x 6144 (8, 8) 40.6 against 45.1 for (8, 5).  The one-block tiles
// are for few rows or columns, where (2, 2) leaves half the CUs idle: two Euler
// steps of 4 layers at hidden 2048 take 484 us against 535 without them at 19
// rows (514 on split-K GEMMs), 500 against 537 (572) at 35; 67 rows at hidden
// 1024 410 against 446 (518).
struct FragTile {
    int nb = 0, mb = 0, ntiles = 0, nms = 0;
};
constexpr int kFragTiles[][2] = {{2, 1}, {2, 2}, {2, 3}, {2, 5}, {4, 1}, {4, 2}, {4, 3}, {4, 4}, {4, 5}, {4, 8}, {8, 4}, {8, 5}, {8, 6}, {8, 8}};
// nb_min, nb_max: bounds from the epilogue.  small: only the tiles up to (4, 5),
// for the operand types that no caller uses above 160 rows (bf16, int8).
FragTile frag_tile(int M, int N, bool small, int nb_min, int nb_max) {
    FragTile best;
    long cost = 0;
    for (const auto& c : kFragTiles) {
        const int nb = c[0], mb = c[1];
        if (nb < nb_min || nb > nb_max || N % (16 * nb) || (small && nb * mb > 20)) continue;
        const int nt = N / (16 * nb), nms = (M + 16 * mb - 1) / (16 * mb);
        const long t = ((long)nt * nms + 255) / 256 * (nb + mb);
        if (!best.nb || t < cost) {
            best.nb = nb;
            best.mb = mb;
            best.ntiles = nt;
            best.nms = nms;
            cost = t;
        }
    }
    return best;
}

struct FragOps {
    const void* a;
    const void* w;
    int K, M;
    bool w8, ah;
    // the rows of a hold x * gamma of a deferred norm
    const float* row_ss;
    int row_tiles;
    float row_inv_n, row_eps;
};

template <int NB, int MB, int U, int NG, bool W8, bool AH, int EPI, int RS>
void launch_frag_one(const FragOps& o, const FragTile& t, const FragEpi& e, hipStream_t s) {
    hipLaunchKernelGGL((gemm_frag_kernel<NB, MB, U, NG, W8, AH, EPI, RS>), dim3(8u * (unsigned)t.nms, (unsigned)((t.ntiles + 7) / 8)),
                       dim3(64 * kFragWaves), 0, s, o.a, o.w, o.K, o.M, t.ntiles, o.row_ss, o.row_tiles, o.row_inv_n,
                       o.row_eps, e);
}

template <int NB, int MB, int U, int NG, bool W8, bool AH, int EPI>
void launch_frag_rows(const FragOps& o, const FragTile& t, const FragEpi& e, hipStream_t s) {
    if constexpr (AH && EPI == SF_EPI_PLAIN) {
        if (o.row_ss) {
            launch_frag_one<NB, MB, U, NG, W8, AH, EPI, kRowGuarded>(o, t, e, s);
            return;
        }
    }
    if constexpr (!AH && EPI != SF_EPI_ADD_NORM) {
        if (o.row_ss) {
            launch_frag_one<NB, MB, U, NG, W8, AH, EPI, kRowDeferred>(o, t, e, s);
            return;
        }
    }
    launch_frag_one<NB, MB, U, NG, W8, AH, EPI, kRowPlain>(o, t, e, s);
}

// U: MFMA steps per group, NG groups: their loads stay within the wave's
// 63-entry load counter and, with the accumulators, its registers.
template <int NB, int MB, int U, int NG, int EPI>
void launch_frag_tile(const FragOps& o, const FragTile& t, const FragEpi& e, hipStream_t s) {
    if constexpr (NB * MB <= 20) {
        if (o.w8) {
            if (o.ah) launch_frag_rows<NB, MB, U / 2, NG, true, true, EPI>(o, t, e, s);
            else launch_frag_rows<NB, MB, U / 2, NG, true, false, EPI>(o, t, e, s);
            return;
        }
        if (!o.ah) {
            launch_frag_rows<NB, MB, U, NG, false, false, EPI>(o, t, e, s);
            return;
        }
    }
    launch_frag_rows<NB, MB, U, NG, false, true, EPI>(o, t, e, s);
}

template <int EPI>
void launch_frag(const FragOps& o, const FragTile& t, const FragEpi& e, hipStream_t s) {
    const int tile = 16 * t.nb + t.mb;
    if constexpr (EPI != SF_EPI_HEADS) {
        switch (tile) {
            case 16 * 2 + 1: launch_frag_tile<2, 1, 8, 2, EPI>(o, t, e, s); return;
            case 16 * 2 + 2: launch_frag_tile<2, 2, 8, 2, EPI>(o, t, e, s); return;
            case 16 * 2 + 3: launch_frag_tile<2, 3, 4, 2, EPI>(o, t, e, s); return;
            case 16 * 2 + 5: launch_frag_tile<2, 5, 4, 2, EPI>(o, t, e, s); return;
            case 16 * 8 + 4: launch_frag_tile<8, 4, 2, 2, EPI>(o, t, e, s); return;
            case 16 * 8 + 5: launch_frag_tile<8, 5, 2, 2, EPI>(o, t, e, s); return;
            case 16 * 8 + 6: launch_frag_tile<8, 6, 2, 2, EPI>(o, t, e, s); return;
            case 16 * 8 + 8: launch_frag_tile<8, 8, 1, 2, EPI>(o, t, e, s); return;
            default: break;
        }
    }
    switch (tile) {
        case 16 * 4 + 1: launch_frag_tile<4, 1, 4, 2, EPI>(o, t, e, s); return;
        case 16 * 4 + 2: launch_frag_tile<4, 2, 4, 2, EPI>(o, t, e, s); return;
        case 16 * 4 + 3: launch_frag_tile<4, 3, 4, 2, EPI>(o, t, e, s); return;
        case 16 * 4 + 4: launch_frag_tile<4, 4, 4, 2, EPI>(o, t, e, s); return;
        case 16 * 4 + 5: launch_frag_tile<4, 5, 2, 2, EPI>(o, t, e, s); return;
        default: launch_frag_tile<4, 8, 2, 2, EPI>(o, t, e, s); return;
    }
}

}  // namespace sfk

namespace {
bool fal16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The tile of a call, its column blocks bounded by the epilogue: a head is one
// tile of 4; the add + norm's tile sums (of 2 column blocks, or of 4 where the
// tile has more) may not exceed what a consumer takes per row.
sfk::FragTile tile_of(const sf_frag_gemm_desc* d, int epilogue) {
    int lo = 2, hi = 8;
    if (epilogue == SF_EPI_HEADS) lo = hi = 4;
    if (epilogue == SF_EPI_ADD_NORM && d->N > 32 * sfk::kFragRowTiles) lo = 4;
    return sfk::frag_tile(d->M, d->N, d->w_dtype == SF_I8 || d->a_dtype != SF_F16, lo, hi);
}
}  // namespace

extern "C" size_t sf_frag_elems(int64_t rows, int64_t cols) {
    return rows > 0 && cols > 0 ? (size_t)((rows + 15) / 16 * 16) * (size_t)cols : 0;
}

extern "C" int32_t sf_gemm_frag_ss_tiles(const sf_frag_gemm_desc* d) {
    if (!d || d->M <= 0 || d->N <= 0) return 0;
    const sfk::FragTile t = tile_of(d, SF_EPI_ADD_NORM);
    return t.nb ? d->N / (16 * std::min(t.nb, 4)) : 0;
}

extern "C" int sf_frag_pack(const sf_frag_job* jobs, int32_t count, void* stream) {
    if (count == 0) return SF_OK;
    if (!jobs || count < 0 || count > SF_CODES_MAX_JOBS) return SF_EINVAL;
    sfk::FragJobs J{};
    J.count = count;
    uint64_t total = 0;
    for (int j = 0; j < count; ++j) {
        const sf_frag_job& b = jobs[j];
        if (b.N < 0 || b.K < 0) return SF_EINVAL;
        const bool i8 = b.w_dtype == SF_I8 && b.out_dtype == SF_I8;
        const bool same = (b.w_dtype == SF_BF16 || b.w_dtype == SF_F16) && b.out_dtype == b.w_dtype;
        const bool cvt = b.w_dtype == SF_BF16 && b.out_dtype == SF_F16;
        const bool widen = b.w_dtype == SF_I8 && b.out_dtype == SF_F16;
        if (!i8 && !same && !cvt && !widen) return SF_ENOTSUP;
        J.start[j] = (uint32_t)total;
        if ((int64_t)b.N * b.K == 0) continue;
        // rows of 16-byte (int8: 8-byte) aligned pieces
        if (!b.w || !b.out || !fal16(b.w) || !fal16(b.out) || (b.N & 15) || (b.K & 63) || b.ldw < b.K || (b.ldw & 7))
            return SF_EINVAL;
        J.w[j] = b.w;
        J.out[j] = b.out;
        J.ldw[j] = b.ldw;
        J.K[j] = b.K;
        J.kind[j] = i8 ? 2 : (widen ? 3 : (cvt ? 1 : 0));
        total += (uint64_t)b.N * (uint64_t)b.K / (i8 ? 16 : 8);
        if (total >= 0x7fffff00ull) return SF_ENOTSUP;   // 32-bit thread indices
    }
    J.start[count] = (uint32_t)total;
    if (total == 0) return SF_OK;
    hipLaunchKernelGGL(sfk::frag_pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), J);
    return hipGetLastError() == hipSuccess ? SF_OK : SF_ELAUNCH;
}

extern "C" int sf_norm_frag(const float* x, int64_t ldx, const float* gamma, void* out, int32_t out_dtype, float* ss,
                            int32_t rows, int32_t cols, float eps, void* stream) {
    if (rows < 0 || cols < 0) return SF_EINVAL;
    if ((long)rows * cols == 0) return SF_OK;
    if (!x || !gamma || !out || ldx < cols) return SF_EINVAL;
    if (out_dtype != SF_BF16 && out_dtype != SF_F16) return SF_ENOTSUP;
    if ((cols & 63) || cols > 2048 * sfk::kNormFragPer) return SF_ENOTSUP;
    if ((ldx & 3) || !fal16(x) || !fal16(gamma) || !fal16(out)) return SF_EINVAL;
    hipLaunchKernelGGL(sfk::norm_frag_kernel, dim3(rows), dim3(256), 0, static_cast<hipStream_t>(stream), x, ldx, gamma,
                       static_cast<uint16_t*>(out), out_dtype == SF_F16 ? 1 : 0, ss, cols, eps, sfk::guard_min(cols));
    return hipGetLastError() == hipSuccess ? SF_OK : SF_ELAUNCH;
}

extern "C" int sf_gemm_frag(const sf_frag_gemm_desc* d, void* stream) {
    if (!d) return SF_EINVAL;
    if (d->M < 0 || d->N < 0 || d->K < 0) return SF_EINVAL;
    if ((long)d->M * d->N == 0) return SF_OK;
    if (d->K == 0 || (d->K & 63) || d->K > (1 << 20) || (d->N & 31)) return SF_ENOTSUP;
    if (d->a_dtype != SF_BF16 && d->a_dtype != SF_F16) return SF_ENOTSUP;
    if (d->w_dtype != d->a_dtype && d->w_dtype != SF_I8) return SF_ENOTSUP;
    if (d->act < 0 || d->act > 2 || (d->act && d->epilogue != SF_EPI_PLAIN)) return SF_EINVAL;
    if (d->a_row_ss && d->epilogue == SF_EPI_ADD_NORM) return SF_EINVAL;
    if (!d->A || !d->W || !fal16(d->A) || !fal16(d->W)) return SF_EINVAL;
    const bool w8 = d->w_dtype == SF_I8;
    if ((w8 && !d->w_scale) || !fal16(d->w_scale)) return SF_EINVAL;
    if (!fal16(d->bias)) return SF_EINVAL;
    // 32-bit byte offsets: a row tile of A, the columns' vectors, all tile sums
    if ((int64_t)128 * d->K * 2 > 0x7fffffffLL || (int64_t)d->N * 4 > 0x7fffffffLL ||
        (int64_t)d->M * sfk::kFragRowTiles * 4 > 0x7fffffffLL)
        return SF_ENOTSUP;
    sfk::FragOps o{d->A, d->W, d->K, d->M, w8, d->a_dtype == SF_F16, nullptr, 0, 0.f, 0.f};
    sfk::FragEpi a{};
    a.w_scale = d->w_scale;
    a.bias = d->bias;
    a.N = d->N;
    a.act = d->act;
    if (d->a_row_ss) {
        if (d->a_row_tiles < 1 || d->a_row_tiles > sfk::kFragRowTiles || d->a_row_n <= 0 || !(d->a_row_eps >= 0.f))
            return SF_EINVAL;
        o.row_ss = d->a_row_ss;
        o.row_tiles = d->a_row_tiles;
        o.row_inv_n = 1.f / (float)d->a_row_n;
        o.row_eps = d->a_row_eps;
        if (d->a_dtype == SF_F16) {   // with the range guard
            if (d->epilogue != SF_EPI_PLAIN || d->a_row_n != d->K) return SF_ENOTSUP;
            if (!d->a_x || !d->a_x_gamma || d->a_x_ld < d->K) return SF_EINVAL;
            a.x = d->a_x;
            a.x_gamma = d->a_x_gamma;
            a.x_ld = d->a_x_ld;
        } else if (d->a_x) {
            return SF_ENOTSUP;
        }
    } else if (d->a_x) {
        return SF_EINVAL;
    }
    const sfk::FragTile t = tile_of(d, d->epilogue);
    if (!t.nb) return SF_ENOTSUP;
    if (d->epilogue == SF_EPI_HEADS) {
        if (d->H <= 0 || d->S <= 0) return SF_EINVAL;
        const int cols = d->H * 64;
        if (d->N % cols || d->N / cols > 3) return SF_EINVAL;
        for (int j = 0; j < d->N / cols; ++j) {
            if (!d->head_out[j] || (reinterpret_cast<uintptr_t>(d->head_out[j]) & 7) || !fal16(d->head_gamma[j]))
                return SF_EINVAL;
            for (int q = 0; q < 3; ++q)
                if (d->head_stride[j][q] & 3) return SF_EINVAL;
            a.head_out[j] = static_cast<uint16_t*>(d->head_out[j]);
            a.head_gamma[j] = d->head_gamma[j];
            a.head_sb[j] = d->head_stride[j][0];
            a.head_sh[j] = d->head_stride[j][1];
            a.head_ss[j] = d->head_stride[j][2];
        }
        a.H = d->H;
        a.S = d->S;
        a.eps = d->eps;
    } else if (d->epilogue == SF_EPI_ADD_NORM) {
        if (!d->C || !fal16(d->C) || d->ldc < d->N || (d->ldc & 3) || d->c_dtype != SF_F32) return SF_EINVAL;
        if (!d->norm_gamma || !fal16(d->norm_gamma) || !d->norm_out || !fal16(d->norm_out) || !d->norm_ss) return SF_EINVAL;
        if (d->norm_dtype != SF_BF16 && d->norm_dtype != SF_F16) return SF_ENOTSUP;
        if (d->N / (16 * std::min(t.nb, 4)) > sfk::kFragRowTiles) return SF_ENOTSUP;
        a.c = d->C;
        a.ldc = d->ldc;
        a.norm_gamma = d->norm_gamma;
        a.norm_out = static_cast<uint16_t*>(d->norm_out);
        a.norm_min = d->norm_dtype == SF_F16 ? sfk::guard_min(d->N) : 0.f;
        a.norm_ss = d->norm_ss;
    } else if (d->epilogue == SF_EPI_PLAIN) {
        if (!d->C) return SF_EINVAL;
        if (d->c_dtype != SF_F32 && d->c_dtype != SF_BF16 && d->c_dtype != SF_F16) return SF_ENOTSUP;
        if (d->accumulate && (d->c_frag || d->c_dtype != SF_F32)) return SF_EINVAL;
        if (d->c_frag) {
            if (d->c_dtype == SF_F32 || !fal16(d->C)) return SF_EINVAL;
        } else if (d->ldc < d->N || (d->ldc & 3) ||
                   (reinterpret_cast<uintptr_t>(d->C) & (d->c_dtype == SF_F32 ? 15u : 7u))) {
            return SF_EINVAL;
        }
        a.c = d->C;
        a.ldc = d->ldc;
        a.c_kind = d->c_dtype == SF_F32 ? 0 : (d->c_dtype == SF_BF16 ? 1 : 2);
        a.c_frag = d->c_frag != 0;
        a.accumulate = d->accumulate != 0;
    } else {
        return SF_ENOTSUP;
    }
    if (a.c && (int64_t)128 * a.ldc * 4 > 0x7fffffffLL) return SF_ENOTSUP;   // 32-bit residual offsets of a row tile
    if ((t.ntiles + 7) / 8 > 65535) return SF_ENOTSUP;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (d->epilogue == SF_EPI_HEADS) sfk::launch_frag<SF_EPI_HEADS>(o, t, a, s);
    else if (d->epilogue == SF_EPI_ADD_NORM) sfk::launch_frag<SF_EPI_ADD_NORM>(o, t, a, s);
    else sfk::launch_frag<SF_EPI_PLAIN>(o, t, a, s);
    return hipGetLastError() == hipSuccess ? SF_OK : SF_ELAUNCH;
}
