// Prefill matmul: C[m, n] = A[m, k] . W (math::matmul, MT:50-74) on the matrix cores.
//
//   f32 weights [n][k]: v_mfma_f32_32x32x2_f32 (full f32 products and accumulation)
//     gemm_f32_small_kernel, gemm_f32_kernel  k % 4 == 0: tiles of 32 to 128 rows, slices of k loaded straight into a ring of LDS regions
//     gemm_f32_any_small_kernel, gemm_f32_any_kernel  any k: 32x32 and 64x64 tiles, register-staged
//   16-bit kernels    bf16 / Q8_0 / Q4_0 weights: v_mfma_f32_32x32x16_{bf16,f16}; activations are
//                     rounded to the matrix-core input type (bf16 for bf16 weights, f16 for
//                     quantised weights, which are expanded to f16(q * d) first).
//     gemm_h256k64_kernel  k % 64 == 0: 256x256 tile, four waves of 128x128, 64-wide k slices
//                          loaded straight into a ring of five LDS regions
//     gemm_narrow_kernel   k % 64 == 0, launches of few tiles: 128 or 256 rows by 64 to 128 columns
//     gemm_h256_kernel     k % 32 == 0: 256x256 tile, eight waves of 128x64, 32-wide slices
//     gemm_h_kernel        any k: 128x128 tile, register-staged
//     gemm_qskinny_kernel  17 to 64 rows on quantised weights: streams the quantised blocks
//     up to 16 rows        the decode matmul's kernels (launch_gemm_few): bf16 with k % 64 == 0 and no infinity, quantised weights with
//                          k % 128 == 0, none of a layered stack with a delta rule
//     gemm_split_reduce_kernel, gemm_tail_reduce_kernel: sums behind launches split along k
#include "device_utils.hpp"
#include <type_traits>

namespace coeus {

constexpr int BM = 64, BN = 64, BK = 32, F32_AHEAD = 3;

// One k slice of both operands for this thread: 2 + 2 pieces of 4 consecutive k (64 rows x 32 k per
// operand = 512 pieces over 256 threads), zero past the edges.
struct F32Slice { float4 a0, a1, w0, w1; };

__device__ __forceinline__ float4 f32_piece(const float *__restrict__ base, uint64_t row, uint64_t rows, uint64_t k, uint64_t kk) {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row >= rows) return v;
    if (kk < k) v.x = base[row * k + kk];
    if (kk + 1 < k) v.y = base[row * k + kk + 1];
    if (kk + 2 < k) v.z = base[row * k + kk + 2];
    if (kk + 3 < k) v.w = base[row * k + kk + 3];
    return v;
}

// Rows that 16-byte pieces do not lie in (k % 4 != 0, or an input that starts between two of them); every other product is gemm_f32_tile's.
template <bool KV>
__global__ __launch_bounds__(256) void gemm_f32_any_kernel(const float *__restrict__ a,
                                                       const float *__restrict__ w, uint64_t m,
                                                       uint64_t n, uint64_t k, EpiArgs e) {
    // k-major tiles: element (row, kk) at [kk][row]; +4 padding keeps the transposing stores
    // and the 32-consecutive-row MFMA operand reads off the same banks.  Two buffers: a slice is
    // written while the previous one is multiplied, one barrier per slice.
    __shared__ float as[2][BK][BM + 4];
    __shared__ float ws[2][BK][BN + 4];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t m0 = (uint64_t)blockIdx.y * BM, n0 = (uint64_t)blockIdx.x * BN;
    const uint32_t wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    float16_t acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.f;

    // piece p = tid + 256 u (u = 0, 1): row p / 8, k offset 4 (p % 8)
    const uint32_t lrow = tid >> 3, lk = (tid & 7) * 4;
    const uint64_t nslices = (k + BK - 1) / BK;
    auto fetch = [&](uint64_t sl) -> F32Slice {
        F32Slice f;
        const uint64_t kk = sl * BK + lk;
        f.a0 = f32_piece(a, m0 + lrow, m, k, kk);
        f.a1 = f32_piece(a, m0 + lrow + 32, m, k, kk);
        f.w0 = f32_piece(w, n0 + lrow, n, k, kk);
        f.w1 = f32_piece(w, n0 + lrow + 32, n, k, kk);
        return f;
    };
    auto put = [&](uint32_t buf, const F32Slice &f) {
        as[buf][lk][lrow] = f.a0.x; as[buf][lk + 1][lrow] = f.a0.y; as[buf][lk + 2][lrow] = f.a0.z; as[buf][lk + 3][lrow] = f.a0.w;
        as[buf][lk][lrow + 32] = f.a1.x; as[buf][lk + 1][lrow + 32] = f.a1.y; as[buf][lk + 2][lrow + 32] = f.a1.z; as[buf][lk + 3][lrow + 32] = f.a1.w;
        ws[buf][lk][lrow] = f.w0.x; ws[buf][lk + 1][lrow] = f.w0.y; ws[buf][lk + 2][lrow] = f.w0.z; ws[buf][lk + 3][lrow] = f.w0.w;
        ws[buf][lk][lrow + 32] = f.w1.x; ws[buf][lk + 1][lrow + 32] = f.w1.y; ws[buf][lk + 2][lrow + 32] = f.w1.z; ws[buf][lk + 3][lrow + 32] = f.w1.w;
    };
    auto mult = [&](uint32_t buf) {
#pragma unroll
        for (int ks = 0; ks < BK; ks += 2) {
            const float fa = as[buf][ks + (lane >> 5)][wm + (lane & 31)];
            const float fb = ws[buf][ks + (lane >> 5)][wn + (lane & 31)];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa, fb, acc, 0, 0, 0);
        }
    };
    // Three slices travel from memory while one is multiplied (small problems are a chain of
    // slices per workgroup: what bounds them is the memory latency per slice, not the bandwidth).
    // Slices past the end come back as zeros.
    F32Slice f0 = fetch(0), f1 = fetch(1), f2 = fetch(2);
    for (uint64_t sl = 0; sl < nslices; sl += F32_AHEAD) {
        put((uint32_t)(sl & 1), f0);
        __syncthreads();
        f0 = fetch(sl + 3);
        mult((uint32_t)(sl & 1));
        if (sl + 1 >= nslices) break;
        put((uint32_t)((sl + 1) & 1), f1);
        __syncthreads();
        f1 = fetch(sl + 4);
        mult((uint32_t)((sl + 1) & 1));
        if (sl + 2 >= nslices) break;
        put((uint32_t)((sl + 2) & 1), f2);
        __syncthreads();
        f2 = fetch(sl + 5);
        mult((uint32_t)((sl + 2) & 1));
    }
    // accumulator i of lane l: row 8*(i/4) + 4*(l/32) + i%4, column l%32
    const uint64_t col = n0 + wn + (lane & 31);
    const bool gated = epi_gated(e.act);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const uint64_t row = m0 + wm + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        // gated: columns (2c, 2c+1) hold (gate_c, up_c) and sit in neighbouring lanes
        const float other = lane_xor1(acc[i]);
        if (row >= m || col >= n) continue;
        if (!gated) epi_store<KV>(e, row, col, acc[i]);
        else if ((lane & 1) == 0) epi_store_gated(e, row, col >> 1, acc[i], other);
    }
}

// The same product for outputs too small to give every CU a 64x64 tile (a prompt of 128 tokens
// has 2 x 12 of them for a 768-wide projection): 32x32 tiles, and the workgroup's four waves split
// every k slice between them (wave v takes k 8v..8v+7 of each 32), so a workgroup's chain of
// slices costs a quarter of the matrix-core time per slice.  A wave fetches and stages exactly the
// 32 x 8 pieces of both operands that it multiplies, in its own part of LDS: no wave waits for
// another inside the loop (LDS serves a wave's stores and loads in order, so there is no barrier
// at all), and each runs six slices of its own requests ahead.  The four partial tiles are added
// through LDS at the end (a different summation order from the 64x64 kernel, the same products).
constexpr int SM = 32, SN = 32, F32S_AHEAD = 6;
struct F32SliceS { float4 a, w; };

template <bool KV>
__global__ __launch_bounds__(256) void gemm_f32_any_small_kernel(const float *__restrict__ a,
                                                             const float *__restrict__ w, uint64_t m,
                                                             uint64_t n, uint64_t k, uint32_t splits, EpiArgs e) {
    __shared__ float as[4][2][8][SM + 4];  // per wave: two buffers of 8 k x 32 rows, k-major
    __shared__ float ws[4][2][8][SN + 4];
    __shared__ float red[4][16][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t m0 = (uint64_t)blockIdx.y * SM, n0 = (uint64_t)blockIdx.x * SN;
    float16_t acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.f;
    const uint32_t lrow = lane >> 1, lk = (lane & 1) * 4;  // the wave's 32 rows x 2 pieces per operand and slice
    // blockIdx.z: this workgroup's share of the slices (a launch split along k stores bare products
    // into plane blockIdx.z of e.out_f32, gemm_split_reduce_kernel sums the planes)
    const uint64_t all_slices = (k + BK - 1) / BK;
    const uint64_t sbeg = all_slices * blockIdx.z / splits, nslices = all_slices * (blockIdx.z + 1) / splits;
    if (splits > 1) e.out_f32 += (uint64_t)blockIdx.z * m * e.n_eff;
    auto fetch = [&](uint64_t sl) -> F32SliceS {
        F32SliceS f;
        f.a = f32_piece(a, m0 + lrow, m, k, sl * BK + 8 * wave + lk);
        f.w = f32_piece(w, n0 + lrow, n, k, sl * BK + 8 * wave + lk);
        return f;
    };
    auto put = [&](uint32_t buf, const F32SliceS &f) {
        float(*pa)[SM + 4] = as[wave][buf];
        float(*pw)[SN + 4] = ws[wave][buf];
        pa[lk][lrow] = f.a.x; pa[lk + 1][lrow] = f.a.y; pa[lk + 2][lrow] = f.a.z; pa[lk + 3][lrow] = f.a.w;
        pw[lk][lrow] = f.w.x; pw[lk + 1][lrow] = f.w.y; pw[lk + 2][lrow] = f.w.z; pw[lk + 3][lrow] = f.w.w;
    };
    auto mult = [&](uint32_t buf) {
#pragma unroll
        for (int ks = 0; ks < 8; ks += 2) {
            const float fa = as[wave][buf][ks + (lane >> 5)][lane & 31];
            const float fb = ws[wave][buf][ks + (lane >> 5)][lane & 31];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa, fb, acc, 0, 0, 0);
        }
    };
    F32SliceS f0 = fetch(sbeg), f1 = fetch(sbeg + 1), f2 = fetch(sbeg + 2), f3 = fetch(sbeg + 3), f4 = fetch(sbeg + 4),
              f5 = fetch(sbeg + 5);
    // (reading a slice's fragments one step ahead of their products, in a register double buffer,
    // changed nothing: a launch is 2 us of launch, 2-3 us until the first operands arrive, 0.14 us per
    // slice of four chained matrix instructions and 1.5 us of epilogue)
#define COEUS_F32S_STEP(F, OFF)                                    \
    if (sl + OFF >= nslices) break;                                \
    put((uint32_t)((sl + OFF) & 1), F);                            \
    F = fetch(sl + OFF + F32S_AHEAD);                              \
    mult((uint32_t)((sl + OFF) & 1));
    for (uint64_t sl = sbeg; sl < nslices; sl += F32S_AHEAD) {
        COEUS_F32S_STEP(f0, 0)
        COEUS_F32S_STEP(f1, 1)
        COEUS_F32S_STEP(f2, 2)
        COEUS_F32S_STEP(f3, 3)
        COEUS_F32S_STEP(f4, 4)
        COEUS_F32S_STEP(f5, 5)
    }
#undef COEUS_F32S_STEP
#pragma unroll
    for (int i = 0; i < 16; i++) red[wave][i][lane] = acc[i];
    __syncthreads();
    // wave v finishes accumulator elements 4v..4v+3: rows 8v + 4 (l / 32) + 0..3, column l % 32
    const uint64_t col = n0 + (lane & 31);
    const bool gated = epi_gated(e.act);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int i = 4 * wave + q;
        const float v = (red[0][i][lane] + red[1][i][lane]) + (red[2][i][lane] + red[3][i][lane]);
        const uint64_t row = m0 + 8 * wave + 4 * (lane >> 5) + q;
        const float other = lane_xor1(v);
        if (row >= m || col >= n) continue;
        if (!gated) epi_store<KV>(e, row, col, v);
        else if ((lane & 1) == 0) epi_store_gated(e, row, col >> 1, v, other);
    }
}

// ---------------------------------------------------------------- 16-bit inputs
// C = A . W^T with A [m][k] and W [n][k] both 16-bit row-major (k contiguous): every lane feeds
// the matrix core 8 consecutive k of one row, for both operands.
constexpr int HM = 128, HN = 128, HK = 32, HLD = 40;  // LDS row stride in elements (80 B)

template <bool BF16>
__global__ __launch_bounds__(256) void gemm_h_kernel(const uint16_t *__restrict__ a,
                                                     const uint16_t *__restrict__ w, uint64_t m,
                                                     uint64_t n, uint64_t k, uint64_t lda,
                                                     uint64_t ldw, EpiArgs e) {
    __shared__ __attribute__((aligned(16))) uint16_t as[HM * HLD];
    __shared__ __attribute__((aligned(16))) uint16_t ws[HN * HLD];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t m0 = (uint64_t)blockIdx.y * HM, n0 = (uint64_t)blockIdx.x * HN;
    const uint32_t wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    float16_t acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[x][y][i] = 0.f;

    const uint32_t lrow = tid >> 1, lseg = (tid & 1) * 16;
    const bool vec = ((k | lda | ldw) & 7) == 0;
    auto load16 = [&](const uint16_t *base, uint64_t ld, uint64_t row, uint64_t rows, uint64_t kk, uint4 &lo, uint4 &hi) {
        lo = make_uint4(0, 0, 0, 0);
        hi = make_uint4(0, 0, 0, 0);
        if (row >= rows) return;
        const uint16_t *p = base + row * ld + kk;
        if (vec) {
            if (kk + 8 <= k) lo = *(const uint4 *)p;
            if (kk + 16 <= k) hi = *(const uint4 *)(p + 8);
        } else {
            uint16_t t[16];
#pragma unroll
            for (int u = 0; u < 16; u++) t[u] = kk + u < k ? p[u] : (uint16_t)0;
            lo = make_uint4(t[0] | (uint32_t)t[1] << 16, t[2] | (uint32_t)t[3] << 16, t[4] | (uint32_t)t[5] << 16, t[6] | (uint32_t)t[7] << 16);
            hi = make_uint4(t[8] | (uint32_t)t[9] << 16, t[10] | (uint32_t)t[11] << 16, t[12] | (uint32_t)t[13] << 16, t[14] | (uint32_t)t[15] << 16);
        }
    };
    uint4 alo, ahi, wlo, whi;
    load16(a, lda, m0 + lrow, m, lseg, alo, ahi);
    load16(w, ldw, n0 + lrow, n, lseg, wlo, whi);
    for (uint64_t k0 = 0; k0 < k; k0 += HK) {
        __syncthreads();
        *(uint4 *)(as + lrow * HLD + lseg) = alo;
        *(uint4 *)(as + lrow * HLD + lseg + 8) = ahi;
        *(uint4 *)(ws + lrow * HLD + lseg) = wlo;
        *(uint4 *)(ws + lrow * HLD + lseg + 8) = whi;
        __syncthreads();
        if (k0 + HK < k) {  // prefetch the next slice while the matrix cores work on this one
            load16(a, lda, m0 + lrow, m, k0 + HK + lseg, alo, ahi);
            load16(w, ldw, n0 + lrow, n, k0 + HK + lseg, wlo, whi);
        }
#pragma unroll
        for (int ks = 0; ks < HK; ks += 16) {
            uint4 af[2], bf[2];
#pragma unroll
            for (int x = 0; x < 2; x++) {
                af[x] = *(const uint4 *)(as + (wm + x * 32 + (lane & 31)) * HLD + ks + 8 * (lane >> 5));
                bf[x] = *(const uint4 *)(ws + (wn + x * 32 + (lane & 31)) * HLD + ks + 8 * (lane >> 5));
            }
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++) {
                    if (BF16) {
                        union { uint4 u; bf16x8_t v; } ua, ub;
                        ua.u = af[x]; ub.u = bf[y];
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ua.v, ub.v, acc[x][y], 0, 0, 0);
                    } else {
                        union { uint4 u; half8_t v; } ua, ub;
                        ua.u = af[x]; ub.u = bf[y];
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ua.v, ub.v, acc[x][y], 0, 0, 0);
                    }
                }
        }
    }
    const bool gated = epi_gated(e.act);
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) {
            const uint64_t col = n0 + wn + y * 32 + (lane & 31);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint64_t row = m0 + wm + x * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                const float other = lane_xor1(acc[x][y][i]);
                if (row >= m || col >= n) continue;
                if (!gated) epi_store(e, row, col, acc[x][y][i]);
                else if ((lane & 1) == 0) epi_store_gated(e, row, col >> 1, acc[x][y][i], other);
            }
        }
}

// ---------------------------------------------------------------- epilogue of the 16-bit matmuls
// Shared by the matmul kernel (accumulators laid out row-major through an LDS strip) and by the
// kernel that sums the partial products of a k-split launch.

// Where 4 consecutive output columns starting at `col` of a prompt pass's q|k|v projection go:
// the key and value thirds are written into the cache (4 consecutive dims of one head).
struct KvCols {
    bool on;
    char *dst;
    uint64_t off;
};
__device__ __forceinline__ KvCols epi_kv_cols(const EpiArgs &e, uint64_t col, uint64_t n) {
    KvCols kc{false, nullptr, 0};
    kc.on = e.kv_k && e.kv_rows_per_seq && col >= e.kv_inner && col + 3 < n;
    if (kc.on) {
        const uint32_t cc = (uint32_t)col;
        const bool is_k = cc < 2 * e.kv_inner;
        const uint32_t c = cc - (is_k ? 1u : 2u) * e.kv_inner, hh = c / e.kv_hd, d = c % e.kv_hd;
        kc.dst = (char *)(is_k ? e.kv_k : e.kv_v);
        kc.off = (uint64_t)hh * e.kv_max_ctx * e.kv_hd + d;
    }
    return kc;
}
__device__ __forceinline__ void epi_store4(const EpiArgs &e, uint64_t row, uint64_t col, const float (&v)[4]) {
    if (e.out_f32) *(float4 *)(e.out_f32 + row * e.n_eff + col) = make_float4(v[0], v[1], v[2], v[3]);
    if (e.out_lp) {
        uint2 p;
        p.x = (uint32_t)f32_to_lp_bits(v[0], e.lp_bf16) | ((uint32_t)f32_to_lp_bits(v[1], e.lp_bf16) << 16);
        p.y = (uint32_t)f32_to_lp_bits(v[2], e.lp_bf16) | ((uint32_t)f32_to_lp_bits(v[3], e.lp_bf16) << 16);
        *(uint2 *)(e.out_lp + row * e.lp_ld + col) = p;
    }
}
// Columns col .. col + 3 of activation row `row` (bias, cache append or activation, residual, store).
// OWN: GELU and SiLU by times_sigmoid where the caller sees f32 results (no further off than the math library's forms), else on the
// hardware's exp2 and reciprocal: at most 17 of 2^-24 off, where the rounding to f16 takes 2^12 of them (root mean square error of a gate to f16 2.0794e-4
// either way; 512 rows of 768 x 3072 with GELU 10.6 us by times_sigmoid, 9.7 on the hardware's).
template <bool OWN = false>
__device__ __forceinline__ void epi_row4(const EpiArgs &e, bool vec4, const KvCols &kc, uint64_t row,
                                         uint64_t col, uint64_t n, float (&v)[4]) {
    if (vec4 && col + 3 < n) {
        if (e.bias) {
            const float4 b4 = *(const float4 *)(e.bias + col);
            v[0] += b4.x; v[1] += b4.y; v[2] += b4.z; v[3] += b4.w;
        }
        if (kc.on) {
            const uint32_t sq = (uint32_t)row / e.kv_rows_per_seq, tok = (uint32_t)row - sq * e.kv_rows_per_seq;
            const uint64_t idx = ((uint64_t)sq * e.kv_heads * e.kv_max_ctx + e.kv_pos0 + tok) * e.kv_hd + kc.off;
            if (e.kv_dtype == COEUS_KV_F32) {
                *(float4 *)((float *)kc.dst + idx) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
                const bool kbf = e.kv_dtype == COEUS_KV_BF16;
                uint2 p;
                p.x = (uint32_t)f32_to_lp_bits(v[0], kbf) | ((uint32_t)f32_to_lp_bits(v[1], kbf) << 16);
                p.y = (uint32_t)f32_to_lp_bits(v[2], kbf) | ((uint32_t)f32_to_lp_bits(v[3], kbf) << 16);
                *(uint2 *)((uint16_t *)kc.dst + idx) = p;
            }
            return;
        }
        if (e.act == COEUS_EPI_GELU)
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = !OWN ? gelu_tanh(v[q]) : e.out_f32 ? gelu_f32(v[q]) : fast_gelu(v[q]);
        if (e.act == COEUS_EPI_SOFTCAP)
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = soft_cap(v[q], e.limit);
        if (e.residual) {
            const float4 r4 = *(const float4 *)(e.residual + row * e.n_eff + col);
            v[0] += r4.x; v[1] += r4.y; v[2] += r4.z; v[3] += r4.w;
        }
        epi_store4(e, row, col, v);
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (col + q < n) epi_store(e, row, col + q, v[q]);
    }
}
// Gated outputs ocol .. ocol + 3 of row `row`, from the weight rows (gate, up) = raw columns
// raw .. raw + 7 (raw = 2 ocol).
template <bool OWN = false>
__device__ __forceinline__ void epi_row4_gated(const EpiArgs &e, bool vec4, uint64_t row, uint64_t ocol,
                                               uint64_t raw, uint64_t n, const float (&gv)[4],
                                               const float (&uv)[4]) {
    if (vec4 && !e.bias && !e.residual && raw + 7 < n) {
        float o[4];
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = e.act == COEUS_EPI_CLAMP_GATE ? clamped_gate(gv[q], uv[q], e.limit) : (!OWN ? silu(gv[q]) : e.out_f32 ? silu_f32(gv[q]) : fast_silu(gv[q])) * uv[q];
        epi_store4(e, row, ocol, o);
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (raw + 2 * q + 1 < n) epi_store_gated(e, row, ocol + q, gv[q], uv[q]);
    }
}

// Sums the partial products of a k-split launch ([splits][m][n] f32, split s holding the products
// over its share of k) in split order and runs the epilogue.  One thread per 4 outputs of a row.
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(const float *__restrict__ part, uint32_t splits,
                                                                uint64_t m, uint64_t n, EpiArgs e) {
    const bool gated = epi_gated(e.act);
    const bool vec4 = e.vec4;
    const uint64_t raw_per_thread = gated ? 8 : 4;
    const uint64_t groups = (n + raw_per_thread - 1) / raw_per_thread;  // per row
    const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= m * groups) return;
    const uint64_t row = gid / groups, raw = (gid - row * groups) * raw_per_thread;
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = 0.f;
    const uint64_t plane = m * n;
    if ((n & 3) == 0) {  // (raw + 3 < n: whole groups of 4)
        for (uint32_t s = 0; s < splits; s++) {
            const float *p = part + s * plane + row * n + raw;
            const float4 a = *(const float4 *)p;
            v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
            if (gated && raw + 7 < n) {
                const float4 c = *(const float4 *)(p + 4);
                v[4] += c.x; v[5] += c.y; v[6] += c.z; v[7] += c.w;
            }
        }
    } else {
        for (uint32_t s = 0; s < splits; s++)
            for (uint64_t q = 0; q < raw_per_thread && raw + q < n; q++) v[q] += part[s * plane + row * n + raw + q];
    }
    if (!gated) {
        float v4[4] = {v[0], v[1], v[2], v[3]};
        epi_row4(e, vec4, epi_kv_cols(e, raw, n), row, raw, n, v4);
    } else {
        const float gv[4] = {v[0], v[2], v[4], v[6]}, uv[4] = {v[1], v[3], v[5], v[7]};
        epi_row4_gated(e, vec4, row, raw >> 1, raw, n, gv, uv);
    }
}

// Which 256x256 output tile the workgroup with number `bid` works on.  Workgroups are numbered so
// that the 32 that run together on one XCD (the hardware deals consecutive workgroups round-robin
// to the 8 XCDs) form a compact block of 4 x 8 output tiles: they walk k in step and share their
// 12 operand tiles through that XCD's L2.
__device__ __forceinline__ void h256_tile_of(uint32_t bid, uint32_t tiles_m, uint32_t tiles_n, uint32_t &tm,
                                             uint32_t &tn) {
    const uint32_t total = tiles_m * tiles_n, per_xcd = total / 8;
    const uint32_t lid = bid < per_xcd * 8 ? (bid % 8) * per_xcd + bid / 8 : bid;
    constexpr uint32_t GM = 4;  // row tiles per group; within a group the order is column-major
    const uint32_t grp = lid / (GM * tiles_n), first_m = grp * GM;
    const uint32_t gsz = min(GM, tiles_m - first_m);
    tm = first_m + (lid % (GM * tiles_n)) % gsz;
    tn = (lid % (GM * tiles_n)) / gsz;
}

// Sums the partial tiles of a launch whose last, incomplete round of tiles was split along k
// ([split][tail tile][256][256] f32) in split order and runs the epilogue.  One thread per 4
// outputs (8 weight rows when gated) of a row; 64 workgroups per tail tile.
__global__ __launch_bounds__(256) void gemm_tail_reduce_kernel(const float *__restrict__ part, uint32_t splits,
                                                               uint32_t full_tiles, uint32_t tiles_m,
                                                               uint32_t tiles_n, uint64_t m, uint64_t n, EpiArgs e) {
    const bool gated = epi_gated(e.act);
    const bool vec4 = e.vec4;
    const uint32_t rpt = gated ? 8 : 4, gpr = 256 / rpt;  // raw columns per thread, threads per tile row
    const uint32_t j = blockIdx.x >> 6, within = (blockIdx.x & 63) * 256 + threadIdx.x;
    const uint32_t r = within / gpr, g = within - r * gpr;
    if (r >= 256) return;
    uint32_t tm, tn;
    h256_tile_of(full_tiles + j, tiles_m, tiles_n, tm, tn);
    const uint64_t row = (uint64_t)tm * 256 + r, raw = (uint64_t)tn * 256 + g * rpt;
    if (row >= m || raw >= n) return;
    const uint32_t tail = tiles_m * tiles_n - full_tiles;
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = 0.f;
    for (uint32_t s = 0; s < splits; s++) {
        const float *p = part + (((uint64_t)s * tail + j) * 256 + r) * 256 + g * rpt;
        const float4 a = *(const float4 *)p;
        v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
        if (gated) {
            const float4 c = *(const float4 *)(p + 4);
            v[4] += c.x; v[5] += c.y; v[6] += c.z; v[7] += c.w;
        }
    }
    if (!gated) {
        float v4[4] = {v[0], v[1], v[2], v[3]};
        epi_row4(e, vec4, epi_kv_cols(e, raw, n), row, raw, n, v4);
    } else {
        const float gv[4] = {v[0], v[2], v[4], v[6]}, uv[4] = {v[1], v[3], v[5], v[7]};
        epi_row4_gated(e, vec4, row, raw >> 1, raw, n, gv, uv);
    }
}

// Large-tile variant for k % 32 == 0 (used when k % 64 != 0; gemm_h256k64_kernel below takes the
// others): 256x256 output tile per workgroup, 8 waves of 128x64
// (8 accumulator tiles of 32x32 per wave; two waves per SIMD, so one wave's LDS waits and
// barriers are covered by the other's matrix-core work).  Per 16-wide k step a wave reads 4 + 2
// operand fragments from LDS for 8 matrix-core instructions.
// The 32-wide k slices go from memory straight into LDS (global_load_lds, 16 bytes per lane, no
// register round trip and no LDS store instructions, which were the bottleneck of a
// register-staged version: LDS stores run at a quarter of the read rate).  Four slice buffers:
// a slice is requested three slices before it is used.  Such a load writes the 64 lanes' pieces
// to 1 KiB of consecutive LDS, which fixes the row stride at 64 bytes; the 16-byte pieces of a
// row are therefore stored XOR-swizzled with bits 2-3 of the row index (the loading lane picks
// the global piece that belongs in its slot), which keeps the 32-row fragment reads spread over
// the banks.  One barrier per slice.
// Workgroups are numbered so that the 32 that run together on one XCD (the hardware deals
// consecutive workgroups round-robin to the 8 XCDs) form a compact block of 4 x 8 output tiles:
// they walk k in step and share their 12 operand tiles through that XCD's L2.
constexpr int TM = 256, TN = 256, TK = 32, NSTAGE = 4;

// Requests one slice: 2 + 2 wave instructions of 1 KiB each, straight into LDS.
__device__ __forceinline__ void slice_request(uint16_t *__restrict__ dst, uint32_t wave,
                                              const uint16_t *const (&ag)[2],
                                              const uint16_t *const (&wg)[2], uint64_t k0) {
    typedef const __attribute__((address_space(1))) void *gptr_t;
    typedef __attribute__((address_space(3))) void *lptr_t;
    uint16_t *as_ = dst + (16 * wave) * TK, *ws_ = as_ + TM * TK;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        __builtin_amdgcn_global_load_lds((gptr_t)(ag[i] + k0), (lptr_t)(as_ + 128 * i * TK), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)(wg[i] + k0), (lptr_t)(ws_ + 128 * i * TK), 16, 0, 0);
    }
}

// One slice of matrix-core work on `sb` while a later slice is requested into `dst`.  The two
// buffers are distinct (__restrict__): that is what lets the fragment reads proceed without
// waiting for the loads into `dst` to land.
template <bool BF16>
__device__ __forceinline__ void slice_step(const uint16_t *__restrict__ sb, uint16_t *__restrict__ dst,
                                           uint32_t wave, const uint16_t *const (&ag)[2],
                                           const uint16_t *const (&wg)[2], uint64_t k_next,
                                           const uint32_t (&afo)[4], const uint32_t (&bfo)[2],
                                           uint32_t fhf, uint32_t fsw, float16_t (&acc)[4][2]) {
    typedef const __attribute__((address_space(1))) void *gptr_t;
    typedef __attribute__((address_space(3))) void *lptr_t;
    uint16_t *as_ = dst + (16 * wave) * TK, *ws_ = as_ + TM * TK;
#pragma unroll
    for (int ks = 0; ks < TK; ks += 16) {
        const uint32_t so = 8 * (((ks >> 3) + fhf) ^ fsw);
        uint4 af[4], bf[2];
        // This wave's four requests for the later slice are spread over the slice, one before each
        // half of a k step's products (all four at the top of the slice measured 5 % slower on
        // the FFN-up shape); they have three slices' time to land.
        const int i = ks >> 4;
        __builtin_amdgcn_global_load_lds((gptr_t)(ag[i] + k_next), (lptr_t)(as_ + 128 * i * TK), 16, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 4; x++) af[x] = *(const uint4 *)(sb + afo[x] + so);
#pragma unroll
        for (int y = 0; y < 2; y++) bf[y] = *(const uint4 *)(sb + bfo[y] + so);
#pragma unroll
        for (int x = 0; x < 4; x++) {
            if (x == 2) {
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_global_load_lds((gptr_t)(wg[i] + k_next), (lptr_t)(ws_ + 128 * i * TK), 16, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int y = 0; y < 2; y++) {
                if (BF16) {
                    union { uint4 u; bf16x8_t v; } ua, ub;
                    ua.u = af[x]; ub.u = bf[y];
                    acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ua.v, ub.v, acc[x][y], 0, 0, 0);
                } else {
                    union { uint4 u; half8_t v; } ua, ub;
                    ua.u = af[x]; ub.u = bf[y];
                    acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ua.v, ub.v, acc[x][y], 0, 0, 0);
                }
            }
        }
    }
}

template <bool BF16>
__global__ __launch_bounds__(512) void gemm_h256_kernel(const uint16_t *a, const uint16_t *w, uint64_t m,
                                                        uint64_t n, uint64_t k, uint64_t lda,
                                                        uint64_t ldw, uint32_t tiles_m,
                                                        uint32_t tiles_n, uint32_t splits, uint32_t full_tiles,
                                                        float *tail_part, EpiArgs e) {
    extern __shared__ __attribute__((aligned(16))) uint16_t sm[];  // [NSTAGE][(TM + TN) * TK]
    constexpr uint32_t BUF = (TM + TN) * TK;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Three kinds of launch:
    //  * plain (splits == 1): workgroup b computes tile b and runs the epilogue;
    //  * every tile split along k (splits > 1, tail_part == nullptr): workgroup b works on tile
    //    b % total over share b / total of the k slices and stores its bare products into plane
    //    b / total of the buffer that e.out_f32 points to ([split][m][n]);
    //  * only the last, incomplete round of tiles split (tail_part != nullptr): workgroups below
    //    full_tiles are plain; the others take tile full_tiles + j over share s of k and store a
    //    whole 256x256 tile of bare products at tail_part[s][j].
    const uint32_t total = tiles_m * tiles_n;
    uint32_t split = 0, bid = blockIdx.x, shares = 1, tail_idx = 0;
    bool tail_wg = false;
    if (tail_part) {
        if (bid >= full_tiles) {
            const uint32_t tail = total - full_tiles, o = bid - full_tiles;
            split = o / tail;
            tail_idx = o - split * tail;
            bid = full_tiles + tail_idx;
            shares = splits;
            tail_wg = true;
        }
    } else if (splits > 1) {
        split = bid / total;
        bid -= split * total;
        shares = splits;
        e.out_f32 += (uint64_t)split * m * e.n_eff;
    }
    const uint64_t nslices = k / TK;
    const uint64_t kbeg = nslices * split / shares * TK, kend = nslices * (split + 1) / shares * TK;
    uint32_t tm, tn;
    h256_tile_of(bid, tiles_m, tiles_n, tm, tn);
    const uint64_t m0 = (uint64_t)tm * TM, n0 = (uint64_t)tn * TN;
    const uint32_t wm = (wave >> 2) * 128, wn = (wave & 3) * 64;
    float16_t acc[4][2];
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[x][y][i] = 0.f;

    // memory -> LDS: a slice is 256 rows x 4 pieces of 16 B per operand.  One wave instruction
    // fills 16 rows (1 KiB); wave v takes rows 16 v + 128 i, lane l row l / 4 of them, slot l % 4,
    // and fetches the piece slot ^ (row / 4 % 4).  Rows past the end are clamped (their results
    // are not stored).
    const uint32_t lr = lane >> 2, lslot = lane & 3;
    const uint16_t *ag[2], *wg[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t row = 16 * wave + 128 * i + lr, piece = lslot ^ ((row >> 2) & 3);
        ag[i] = a + (m0 + min((uint64_t)row, m - 1 - m0)) * lda + piece * 8;
        wg[i] = w + (n0 + min((uint64_t)row, n - 1 - n0)) * ldw + piece * 8;
    }
    const uint64_t klast = kend - TK;
    slice_request(sm, wave, ag, wg, kbeg);
    slice_request(sm + BUF, wave, ag, wg, kbeg + TK <= klast ? kbeg + TK : klast);
    slice_request(sm + 2 * BUF, wave, ag, wg, kbeg + 2 * TK <= klast ? kbeg + 2 * TK : klast);
    __builtin_amdgcn_s_waitcnt(0x0078);  // vmcnt(8): slice 0 has landed (this wave's part)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t frow = lane & 31, fhf = lane >> 5;
    // fragment addresses (elements) within a slice buffer: row * 32 + 8 * (piece ^ (row / 4 % 4))
    uint32_t afo[4], bfo[2];
#pragma unroll
    for (int x = 0; x < 4; x++) afo[x] = (wm + x * 32 + frow) * TK;
#pragma unroll
    for (int y = 0; y < 2; y++) bfo[y] = (TM + wn + y * 32 + frow) * TK;
    const uint32_t fsw = (frow >> 2) & 3;  // the same for every fragment row of a lane: tiles start at multiples of 32
    uint32_t st = 0;
    for (uint64_t k0 = kbeg; k0 < kend; k0 += TK) {
        // slice k0 + 3 TK goes into the buffer whose slice (k0 - TK) everybody finished before the
        // last barrier; past the end the last slice is requested again and never used
        slice_step<BF16>(sm + st * BUF, sm + ((st + 3) & (NSTAGE - 1)) * BUF, wave, ag, wg,
                         k0 + 3 * TK <= klast ? k0 + 3 * TK : klast, afo, bfo, fhf, fsw, acc);
        // The next slice has landed (this wave's part: all but the 8 newest loads are done) and
        // this wave's fragment reads are done; then the workgroup barrier.  Not __syncthreads():
        // its fence would wait for every load in flight.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0x0078);  // vmcnt(8) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        st = (st + 1) & (NSTAGE - 1);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): nothing may land in LDS once it is reused below

    // Epilogue through LDS (free now): each wave lays one 32-row strip of its 128x64 block at a
    // time out row-major in a private [32][64 + 4] area and walks it with 16-byte accesses: a
    // store instruction covers four 256-byte row segments, and the epilogue is a short loop
    // instead of 128 unrolled scalar copies.
    constexpr uint32_t TS = 68;
    float *strip = (float *)sm + wave * (32 * TS);
    // where the epilogue writes: the output matrix, or (tail workgroups) a private 256x256 tile
    uint64_t em = m, en = n, em0 = m0, en0 = n0;
    if (tail_wg) {
        EpiArgs pe = {};
        pe.out_f32 = tail_part + ((uint64_t)split * (total - full_tiles) + tail_idx) * (TM * TN);
        pe.n = pe.n_eff = TN;
        pe.vec4 = 1;
        e = pe;
        em = TM; en = TN; em0 = 0; en0 = 0;
    }
    const bool gated = epi_gated(e.act);
    const bool vec4 = e.vec4;
    auto strip_out = [&](const float16_t (&t)[2], uint32_t x) {
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                strip[(8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)) * TS + y * 32 + (lane & 31)] = t[y][i];
        const uint64_t row0 = em0 + wm + x * 32, col0 = en0 + wn;
        if (!gated) {
            const uint32_t c4 = (lane & 15) * 4;
            const KvCols kc = epi_kv_cols(e, col0 + c4, en);
#pragma unroll 2
            for (uint32_t r = lane >> 4; r < 32; r += 4) {
                const uint64_t row = row0 + r, col = col0 + c4;
                const float4 v4 = *(const float4 *)(strip + r * TS + c4);
                float v[4] = {v4.x, v4.y, v4.z, v4.w};
                if (row >= em) continue;
                epi_row4(e, vec4, kc, row, col, en, v);
            }
        } else {
            // weight rows (2c, 2c+1) = (gate_c, up_c): a lane takes 4 outputs = 8 strip columns
            const uint32_t o4 = (lane & 7) * 4;
#pragma unroll 2
            for (uint32_t r = lane >> 3; r < 32; r += 8) {
                const uint64_t row = row0 + r, ocol = (col0 >> 1) + o4;
                const float4 p0 = *(const float4 *)(strip + r * TS + 2 * o4);
                const float4 p1 = *(const float4 *)(strip + r * TS + 2 * o4 + 4);
                const float gv[4] = {p0.x, p0.z, p1.x, p1.z}, uv[4] = {p0.y, p0.w, p1.y, p1.w};
                if (row >= em) continue;
                epi_row4_gated(e, vec4, row, ocol, col0 + 2 * o4, en, gv, uv);
            }
        }
    };
    __syncthreads();  // every wave has finished reading the operand slices, every load has landed
    strip_out(acc[0], 0);
    strip_out(acc[1], 1);
    strip_out(acc[2], 2);
    strip_out(acc[3], 3);
}

// The same 256x256 tile for k % 64 == 0, built around what a CU's shared resources cost per 64 of
// k: 2048 cycles of matrix-core work per SIMD; LDS fragment reads (1024 cycles' worth with eight
// waves of 128x64, 512 with four waves of 128x128); and the path from L2 into LDS, which moves
// whole 128-byte lines whether a request asks for 64 or 128 bytes of them and needs three quarters
// of the matrix-core time for a slice even when nothing else runs.  So: four waves of 128x128
// (16 accumulator tiles each in the accumulation registers, one wave per SIMD), 64-wide k slices,
// loads into LDS that take 8 rows x 128 bytes per wave instruction (full lines), and a schedule
// in which the loads go out one behind every fourth product, all through the slice, each with
// one and a half to two slice times to land.
//
// LDS (160 KiB): three 32-KiB regions for the A rows of a slice, two for the W rows; slice s uses
// A region s % 3 and W region s % 2.  Row stride 128 bytes, the eight 16-byte pieces of a row
// stored at slot = piece ^ (row / 2 % 8) (with row % 8 half of the LDS cycles of the 32-row
// fragment reads are bank conflicts, with row / 2 % 8 none).
//
// A wave keeps the W fragments of the whole slice in registers (4 column blocks x 4 k steps) and
// walks its four 32-row blocks of A one after the other ("step" x: 16 products, 4 k steps x 4
// column blocks, on the A fragments of row block x).  That frees the W region as soon as the
// fragments are read.  One period of the loop runs from the barrier before a slice's last step
// to the next such barrier:
//   step 3 of slice s     reads the A fragments of step 0 and, k step by k step as the old ones
//                         retire, the W fragments of slice s + 1; requests A rows of slice s + 3
//                         into the region that slice s has finished with (barrier 1)
//   step 0 of slice s + 1 reads the A fragments of step 1; the rest of those requests
//   barrier 2             every wave holds the W fragments of slice s + 1: their region is free
//   steps 1 and 2         read the A fragments of steps 2 and 3; request the W rows of slice s + 3
//   barrier 1             behind it the loads of slice s + 2 have landed for every wave (all but
//                         the 16 newest requests of a wave are done)
// Nothing else runs on a wave's SIMD, so every wait is placed where it is already satisfied, and
// the waits are explicit: next to a pending load into LDS the compiler turns a wait for one
// fragment into a wait for all reads.
constexpr int UK = 64;
constexpr uint32_t UREG = 256 * UK;  // elements per region

struct K64Frags {
    uint4 a[2][4];  // [buffer][k step]: the A fragments of one row block
    uint4 b[4][4];  // [column block][k step]: the W fragments of a slice
};

template <bool BF16>
__device__ __forceinline__ void mfma_32x32x16(const uint4 &a, const uint4 &b, float16_t &c) {
    if (BF16) {
        union { uint4 u; bf16x8_t v; } ua, ub;
        ua.u = a; ub.u = b;
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ua.v, ub.v, c, 0, 0, 0);
    } else {
        union { uint4 u; half8_t v; } ua, ub;
        ua.u = a; ub.u = b;
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ua.v, ub.v, c, 0, 0, 0);
    }
}

// Where the loads of a wave come from: unit 4 q + wave of an operand is 8 rows x 128 bytes; lane
// l takes row l / 8 of them and the piece that belongs in slot l % 8.  Rows past the end are
// clamped (their results are not stored).  The address is a uniform base plus a 32-bit lane
// offset, so a request costs one vector addition between two products.
struct K64Source {
    const char *a, *w;      // tile origins (uniform)
    uint32_t oa[8], ow[8];  // this lane's byte offsets for the wave's eight units of each operand
};

__device__ __forceinline__ void k64_request(const K64Source &src, int q, bool is_w, uint64_t k0, uint16_t *region,
                                            uint32_t wave) {
    typedef const __attribute__((address_space(1))) void *gptr_t;
    typedef __attribute__((address_space(3))) void *lptr_t;
    const char *p = (is_w ? src.w : src.a) + 2 * k0 + (uint64_t)(is_w ? src.ow[q] : src.oa[q]);
    __builtin_amdgcn_global_load_lds((gptr_t)p, (lptr_t)(region + (4 * q + wave) * 512), 16, 0, 0);
}

// Lane constants of the fragment reads (elements): row * 64 + 8 * (piece ^ (row / 2 % 8)) with
// piece = 2 (k step) + lane / 32; a lane's rows are all congruent to lane % 32 modulo 32.
struct K64Lane {
    uint32_t a[4], w[4];  // [k step], row block 0 / column block 0 of the wave
};

__device__ __forceinline__ uint4 k64_read(const uint16_t *region, uint32_t lane_off, int block) {
    return *(const uint4 *)(region + lane_off + block * (32 * UK));
}

// One period (see above).  HEAD: the first slice of a tile: no step 3 in front, the fragments of
// its step 0 and all its W fragments are already in registers.  REQUEST: slice s + 3 exists.
// rd_a / rd_w: regions of slice s + 1; free_a: region of slice s (gets A of s + 3); rd_w is also
// where W of s + 3 goes, after barrier 2: the restrict qualifiers tell the compiler that reads
// never have to wait for loads in flight, which holds because the barriers order them.
template <bool BF16, bool HEAD, bool REQUEST>
__device__ __forceinline__ void k64_period(const uint16_t *__restrict__ rd_a, const uint16_t *__restrict__ rd_w,
                                           uint16_t *__restrict__ free_a, uint16_t *__restrict__ free_w,
                                           const K64Lane &ln, uint32_t wave, const K64Source &src, uint64_t k_req,
                                           K64Frags &f, float16_t (&acc)[4][4]) {
    if (!HEAD) {
        // step 3 of slice s: reads #1-4 A of step 0 (gaps 0-2), #5-17 W of slice s + 1 (gaps 3-15)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int kk = i >> 2, y = i & 3;
            mfma_32x32x16<BF16>(f.b[y][kk], f.a[1][kk], acc[3][y]);
            if (i == 15) __builtin_amdgcn_s_waitcnt(0xC87F);  // lgkmcnt(8): reads #1-8 (step 0, k step 0) are there
            if (i < 3) f.a[0][i] = k64_read(rd_a, ln.a[i], 0);
            if (i == 2) f.a[0][3] = k64_read(rd_a, ln.a[3], 0);
            if (i >= 3) f.b[(i - 3) & 3][(i - 3) >> 2] = k64_read(rd_w, ln.w[(i - 3) >> 2], (i - 3) & 3);
            if (REQUEST && (i & 3) == 1) k64_request(src, i >> 2, false, k_req, free_a, wave);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // step 0 of slice s + 1: reads #18-20 the last W fragments (gaps 0-2), #21-24 A of step 1 (gaps 3-6)
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int kk = i >> 2, y = i & 3;
        if (!HEAD && i == 12) {
            __builtin_amdgcn_s_waitcnt(0xC47F);  // lgkmcnt(4): reads #17-20 (k step 3) are there
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_nop 0");
        }
        mfma_32x32x16<BF16>(f.b[y][kk], f.a[0][kk], acc[0][y]);
        if (!HEAD && i == 3) __builtin_amdgcn_s_waitcnt(0xC87F);  // lgkmcnt(8): 20 issued, #9-12 (k step 1) are there
        if (!HEAD && i == 6) __builtin_amdgcn_s_waitcnt(0xC77F);  // lgkmcnt(7): 23 issued, #13-16 (k step 2) are there
        if (!HEAD && i < 3) f.b[i + 1][3] = k64_read(rd_w, ln.w[3], i + 1);
        if (i >= 3 && i < 7) f.a[1][i - 3] = k64_read(rd_a, ln.a[i - 3], 1);
        if (REQUEST && !HEAD && (i & 3) == 1) k64_request(src, 4 + (i >> 2), false, k_req, free_a, wave);
        __builtin_amdgcn_sched_barrier(0);
    }
    // barrier 2: every wave has its W fragments of slice s + 1 (it has used them all)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the A fragments of step 1 are there
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int kk = i >> 2, y = i & 3;
        mfma_32x32x16<BF16>(f.b[y][kk], f.a[1][kk], acc[1][y]);
        if (i < 4) f.a[0][i] = k64_read(rd_a, ln.a[i], 2);
        if (REQUEST && (i & 3) == 1) k64_request(src, i >> 2, true, k_req, free_w, wave);
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the A fragments of step 2 are there
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int kk = i >> 2, y = i & 3;
        mfma_32x32x16<BF16>(f.b[y][kk], f.a[0][kk], acc[2][y]);
        if (i < 4) f.a[1][i] = k64_read(rd_a, ln.a[i], 3);
        if (REQUEST && (i & 3) == 1) k64_request(src, 4 + (i >> 2), true, k_req, free_w, wave);
        __builtin_amdgcn_sched_barrier(0);
    }
    // barrier 1: the A fragments of step 3 are there, so this wave has no read of slice s + 1 in
    // flight; its loads of slice s + 2 have landed (all but this period's 16, or all)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (REQUEST) __builtin_amdgcn_s_waitcnt(0x4070);  // vmcnt(16) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0070);          // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_sched_barrier(0);
}

// Epilogue: 32 rows x 128 columns of a wave's block at a time go through a private
// [32][128 + 4] LDS area and out in 16-byte accesses (in both directions: the weight fragment is
// the first operand of the products, so a lane holds row lane % 32 of the block and, per register
// group g, the 4 consecutive columns 8 g + 4 (lane / 32) ...).
constexpr uint32_t K64_TS = 132;

__device__ __forceinline__ void k64_strip_write(float *strip, const float16_t (&t)[4], uint32_t lane) {
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            *(float4 *)(strip + (lane & 31) * K64_TS + y * 32 + 8 * g + 4 * (lane >> 5)) =
                make_float4(t[y][4 * g], t[y][4 * g + 1], t[y][4 * g + 2], t[y][4 * g + 3]);
}

// (the 16-bit type is a template parameter: chosen at run time per value, both conversions are
// computed for every value)
template <bool BF16OUT>
__device__ __forceinline__ uint2 k64_pack4(const float (&v)[4]) {
    uint2 p;
    p.x = (uint32_t)f32_to_lp_bits(v[0], BF16OUT) | ((uint32_t)f32_to_lp_bits(v[1], BF16OUT) << 16);
    p.y = (uint32_t)f32_to_lp_bits(v[2], BF16OUT) | ((uint32_t)f32_to_lp_bits(v[3], BF16OUT) << 16);
    return p;
}

// Any epilogue, decided value by value (blocks that end outside the matrix, unusual layouts).
__device__ __forceinline__ void k64_strip_generic(const float *strip, uint32_t lane, const EpiArgs &e, bool gated,
                                                  bool vec4, uint64_t row0, uint64_t col0, uint64_t em, uint64_t en) {
    if (!gated) {
        const uint32_t c4 = (lane & 31) * 4;
        const KvCols kc = epi_kv_cols(e, col0 + c4, en);
#pragma unroll 2
        for (uint32_t r = lane >> 5; r < 32; r += 2) {
            const uint64_t row = row0 + r, col = col0 + c4;
            const float4 v4 = *(const float4 *)(strip + r * K64_TS + c4);
            float v[4] = {v4.x, v4.y, v4.z, v4.w};
            if (row >= em) continue;
            epi_row4(e, vec4, kc, row, col, en, v);
        }
    } else {
        // weight rows (2c, 2c+1) = (gate_c, up_c): a lane takes 4 outputs = 8 strip columns
        const uint32_t o4 = (lane & 15) * 4;
#pragma unroll 2
        for (uint32_t r = lane >> 4; r < 32; r += 4) {
            const uint64_t row = row0 + r, ocol = (col0 >> 1) + o4;
            const float4 p0 = *(const float4 *)(strip + r * K64_TS + 2 * o4);
            const float4 p1 = *(const float4 *)(strip + r * K64_TS + 2 * o4 + 4);
            const float gv[4] = {p0.x, p0.z, p1.x, p1.z}, uv[4] = {p0.y, p0.w, p1.y, p1.w};
            if (row >= em) continue;
            epi_row4_gated(e, vec4, row, ocol, col0 + 2 * o4, en, gv, uv);
        }
    }
}

// The activations of the 16-bit matmuls' fast walks, on the hardware's exp2 and reciprocal (1 ulp
// each; tanhf, expf and the division cost 4-5 times the instructions, and a SiLU-gated block
// evaluates 128 of them per lane): x * sigmoid(x), and 0.5 x (1 + tanh(u)) = x * sigmoid(2 u).
__device__ __forceinline__ float k64_sigmoid(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}
__device__ __forceinline__ float k64_silu(float x) { return x * k64_sigmoid(x); }
__device__ __forceinline__ float k64_gelu(float x) {
    const float c0 = 0.7978845608028654f, c1 = 0.044715f;
    return x * k64_sigmoid(2.0f * c0 * x * (1.0f + c1 * x * x));
}

// The common epilogues with every decision made outside the loop over rows (the generic walk
// takes some 400 cycles per 16-byte store, a fifth of a 4096-long tile's time in all).  All 128
// columns of the block lie inside the matrix and 4-column accesses are aligned.  A lane takes
// columns 4 (lane % 32) ... + 3 of rows lane / 32, + 2, ...; the residual values of a strip are
// all requested before its first store goes out (a wait for a load behind a store would wait for
// that store to be acknowledged as well).
template <bool BIAS, bool RES, bool GELU, bool LP, bool BF16OUT = false>
__device__ __forceinline__ void k64_strip_rows(const float *strip, uint32_t lane, const EpiArgs &e, uint64_t row0,
                                               uint64_t col0, uint64_t em) {
    const uint32_t c4 = (lane & 31) * 4, r0 = lane >> 5;
    const uint64_t col = col0 + c4;
    float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (BIAS) b4 = *(const float4 *)(e.bias + col);
    const float *sp = strip + r0 * K64_TS + c4;
    const uint64_t ld = LP ? e.lp_ld : e.n_eff;
    uint64_t row = row0 + r0;
    const float *rp = RES ? e.residual + row * e.n_eff + col : nullptr;
    float *of = LP ? nullptr : e.out_f32 + row * ld + col;
    uint16_t *ol = LP ? e.out_lp + row * ld + col : nullptr;
    // groups of 8 rows (the residual values of a group are requested before its stores)
#pragma unroll 1
    for (int jj = 0; jj < 2; jj++) {
        float4 res[8];
        if (RES) {
#pragma unroll
            for (int j = 0; j < 8; j++)
                res[j] = row + 2 * j < em ? *(const float4 *)(rp + (uint64_t)(2 * j) * e.n_eff) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float4 v4 = *(const float4 *)(sp + 2 * j * K64_TS);
            float v[4] = {v4.x + b4.x, v4.y + b4.y, v4.z + b4.z, v4.w + b4.w};
            if (GELU)
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = k64_gelu(v[q]);
            if (RES) { v[0] += res[j].x; v[1] += res[j].y; v[2] += res[j].z; v[3] += res[j].w; }
            if (row + 2 * j < em) {
                if (LP) *(uint2 *)(ol + (uint64_t)(2 * j) * ld) = k64_pack4<BF16OUT>(v);
                else *(float4 *)(of + (uint64_t)(2 * j) * ld) = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        sp += 16 * K64_TS;
        row += 16;
        if (RES) rp += 16 * e.n_eff;
        if (LP) ol += 16 * ld; else of += 16 * ld;
    }
}

// The residual epilogue (h += ...: f32 in, f32 out) of a whole 128x128 block.  Waiting for a
// strip's 16 KiB of residual values strip by strip, each wait behind the previous strip's stores,
// took 60 k cycles per tile, over a third of a 4096-long tile's matmul time.  Here the values of
// strip x + 2 are requested when strip x has been stored, into the registers that strip x's values
// occupied (the fragment registers are free by now), so every request has a strip's time to land
// and no wait for a load is also a wait for younger stores.
template <bool BIAS>
__device__ __forceinline__ void k64_epilogue_residual(float *strip, float16_t (&acc)[4][4], uint32_t lane,
                                                      const EpiArgs &e, uint64_t row0, uint64_t col0, uint64_t em) {
    const uint32_t c4 = (lane & 31) * 4, r0 = lane >> 5;
    const uint64_t col = col0 + c4;
    float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (BIAS) b4 = *(const float4 *)(e.bias + col);
    float4 res[2][16];
    auto request = [&](int x, float4 (&r)[16]) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const uint64_t row = row0 + 32 * x + r0 + 2 * j;
            r[j] = row < em ? *(const float4 *)(e.residual + row * e.n_eff + col) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    request(0, res[0]);
    request(1, res[1]);
#pragma unroll
    for (int x = 0; x < 4; x++) {
        k64_strip_write(strip, acc[x], lane);
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const uint32_t r = r0 + 2 * j;
            const uint64_t row = row0 + 32 * x + r;
            const float4 v4 = *(const float4 *)(strip + r * K64_TS + c4);
            const float4 q = res[x & 1][j];
            if (row < em)
                *(float4 *)(e.out_f32 + row * e.n_eff + col) =
                    make_float4(v4.x + b4.x + q.x, v4.y + b4.y + q.y, v4.z + b4.z + q.z, v4.w + b4.w + q.w);
        }
        if (x + 2 < 4) request(x + 2, res[x & 1]);
    }
}

// Key / value columns of a prompt pass's q|k|v projection: straight into the cache.
template <bool BIAS, int KVT>  // KVT: COEUS_KV_F32 / F16 / BF16
__device__ __forceinline__ void k64_strip_kv(const float *strip, uint32_t lane, const EpiArgs &e, uint64_t row0,
                                             uint64_t col0, uint64_t em, uint64_t en) {
    const uint32_t c4 = (lane & 31) * 4, r0 = lane >> 5;
    const uint64_t col = col0 + c4;
    const KvCols kc = epi_kv_cols(e, col, en);
    float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (BIAS) b4 = *(const float4 *)(e.bias + col);
    // sequence and token of the strip's first row; rows advance by 2 per step
    uint32_t sq = (uint32_t)(row0 + r0) / e.kv_rows_per_seq, tok = (uint32_t)(row0 + r0) - sq * e.kv_rows_per_seq;
#pragma unroll 4
    for (int j = 0; j < 16; j++) {
        const uint32_t r = r0 + 2 * j;
        const float4 v4 = *(const float4 *)(strip + r * K64_TS + c4);
        const float v[4] = {v4.x + b4.x, v4.y + b4.y, v4.z + b4.z, v4.w + b4.w};
        if (row0 + r < em) {
            const uint64_t idx = ((uint64_t)sq * e.kv_heads * e.kv_max_ctx + e.kv_pos0 + tok) * e.kv_hd + kc.off;
            if (KVT == COEUS_KV_F32) *(float4 *)((float *)kc.dst + idx) = make_float4(v[0], v[1], v[2], v[3]);
            else *(uint2 *)((uint16_t *)kc.dst + idx) = k64_pack4<KVT == COEUS_KV_BF16>(v);
        }
        tok += 2;
        while (tok >= e.kv_rows_per_seq) { tok -= e.kv_rows_per_seq; sq++; }
    }
}

// Gated pairs without bias or residual: weight rows (2c, 2c+1) = (gate_c, up_c); a lane
// takes 4 outputs = 8 strip columns of rows lane / 16, + 4, ...
template <bool CLAMP, bool LP, bool BF16OUT = false>
__device__ __forceinline__ void k64_strip_gated(const float *strip, uint32_t lane, const EpiArgs &e, uint64_t row0,
                                                uint64_t col0, uint64_t em) {
    const uint32_t o4 = (lane & 15) * 4, r0 = lane >> 4;
    const uint64_t ocol = (col0 >> 1) + o4;
#pragma unroll 4
    for (int j = 0; j < 8; j++) {
        const uint32_t r = r0 + 4 * j;
        const uint64_t row = row0 + r;
        const float4 p0 = *(const float4 *)(strip + r * K64_TS + 2 * o4);
        const float4 p1 = *(const float4 *)(strip + r * K64_TS + 2 * o4 + 4);
        float v[4];
        if (CLAMP) {
            v[0] = clamped_gate(p0.x, p0.y, e.limit); v[1] = clamped_gate(p0.z, p0.w, e.limit);
            v[2] = clamped_gate(p1.x, p1.y, e.limit); v[3] = clamped_gate(p1.z, p1.w, e.limit);
        } else {
            v[0] = k64_silu(p0.x) * p0.y; v[1] = k64_silu(p0.z) * p0.w;
            v[2] = k64_silu(p1.x) * p1.y; v[3] = k64_silu(p1.z) * p1.w;
        }
        if (row < em) {
            if (LP) *(uint2 *)(e.out_lp + row * e.lp_ld + ocol) = k64_pack4<BF16OUT>(v);
            else *(float4 *)(e.out_f32 + row * e.n_eff + ocol) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

// The same to 16 bits straight from the accumulators: a lane holds row lane % 32 of a 32 x 32 block and, per register group g, the
// pairs of outputs 4 g + 2 (lane / 32) and + 1.  Packed, two swaps with the lane that has the row's other outputs leave 16
// consecutive bytes a lane, 32 a row: no trip through LDS (7B shape, 4071 rows, whole pass 51.8 -> 51.1 ms).  Rows without a
// gate are better off through LDS, where a store covers 256 bytes of a row (1B shape with GELU 44.8 -> 45.2 ms this way).
template <bool CLAMP, bool BF16OUT>
__device__ __forceinline__ void k64_direct_gated(const float16_t (&t)[4], uint32_t lane, const EpiArgs &e, uint64_t row, uint64_t col0,
                                                 uint64_t em) {
    uint16_t *out = e.out_lp + row * e.lp_ld + (col0 >> 1) + 8 * (lane >> 5);
#pragma unroll
    for (int y = 0; y < 4; y++) {
        uint32_t p[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float g0 = t[y][4 * g], u0 = t[y][4 * g + 1], g1 = t[y][4 * g + 2], u1 = t[y][4 * g + 3];
            const float a = CLAMP ? clamped_gate(g0, u0, e.limit) : k64_silu(g0) * u0, b = CLAMP ? clamped_gate(g1, u1, e.limit) : k64_silu(g1) * u1;
            p[g] = (uint32_t)f32_to_lp_bits(a, BF16OUT) | ((uint32_t)f32_to_lp_bits(b, BF16OUT) << 16);
        }
        const auto lo = __builtin_amdgcn_permlane32_swap(p[0], p[2], false, false), hi = __builtin_amdgcn_permlane32_swap(p[1], p[3], false, false);
        if (row < em) *(uint4 *)(out + y * 16) = make_uint4(lo[0], lo[1], hi[0], hi[1]);
    }
}

// Which of the walks above serves a wave's block: decided once per block.
enum : uint32_t { K64_GENERIC = 0, K64_ROWS = 1, K64_KV = 2, K64_GATED = 3 };
// for K64_ROWS the low bits of `bits` select bias (1), residual (2), GELU (4), 16-bit output (8)
__device__ __forceinline__ uint32_t k64_epilogue_kind(const EpiArgs &e, bool vec4, uint64_t col0, uint64_t en,
                                                      uint32_t &bits) {
    bits = (e.bias ? 1u : 0u) | (e.residual ? 2u : 0u) | (e.act == COEUS_EPI_GELU ? 4u : 0u) | (e.out_lp ? 8u : 0u);
    const bool one_out = (e.out_f32 != nullptr) != (e.out_lp != nullptr);
    if (!vec4 || col0 + 128 > en || (en & 3)) return K64_GENERIC;
    if (e.act == COEUS_EPI_SOFTCAP) return K64_GENERIC;
    if (epi_gated(e.act)) return (!e.bias && !e.residual && one_out) ? K64_GATED : K64_GENERIC;
    if (e.kv_k) {
        if (!e.kv_rows_per_seq || (e.kv_inner & 127)) return K64_GENERIC;
        if (col0 >= e.kv_inner) return K64_KV;
    }
    if (!one_out || (e.residual && e.out_lp) || (bits & 4 && bits & 2)) return K64_GENERIC;
    return K64_ROWS;
}

__device__ __forceinline__ void k64_strip_out(const float *strip, uint32_t lane, const EpiArgs &e, uint32_t kind,
                                              uint32_t bits, bool gated, bool vec4, uint64_t row0, uint64_t col0,
                                              uint64_t em, uint64_t en) {
    if (kind == K64_ROWS) {
        switch (bits) {
        case 0: k64_strip_rows<false, false, false, false>(strip, lane, e, row0, col0, em); break;
        case 1: k64_strip_rows<true, false, false, false>(strip, lane, e, row0, col0, em); break;
        case 2: k64_strip_rows<false, true, false, false>(strip, lane, e, row0, col0, em); break;
        case 3: k64_strip_rows<true, true, false, false>(strip, lane, e, row0, col0, em); break;
        case 4: k64_strip_rows<false, false, true, false>(strip, lane, e, row0, col0, em); break;
        case 5: k64_strip_rows<true, false, true, false>(strip, lane, e, row0, col0, em); break;
        case 8:
            if (e.lp_bf16) k64_strip_rows<false, false, false, true, true>(strip, lane, e, row0, col0, em);
            else k64_strip_rows<false, false, false, true, false>(strip, lane, e, row0, col0, em);
            break;
        case 9:
            if (e.lp_bf16) k64_strip_rows<true, false, false, true, true>(strip, lane, e, row0, col0, em);
            else k64_strip_rows<true, false, false, true, false>(strip, lane, e, row0, col0, em);
            break;
        case 12:
            if (e.lp_bf16) k64_strip_rows<false, false, true, true, true>(strip, lane, e, row0, col0, em);
            else k64_strip_rows<false, false, true, true, false>(strip, lane, e, row0, col0, em);
            break;
        case 13:
            if (e.lp_bf16) k64_strip_rows<true, false, true, true, true>(strip, lane, e, row0, col0, em);
            else k64_strip_rows<true, false, true, true, false>(strip, lane, e, row0, col0, em);
            break;
        default: k64_strip_generic(strip, lane, e, gated, vec4, row0, col0, em, en); break;
        }
    } else if (kind == K64_KV) {
        if (e.kv_dtype == COEUS_KV_F16) {
            if (e.bias) k64_strip_kv<true, COEUS_KV_F16>(strip, lane, e, row0, col0, em, en);
            else k64_strip_kv<false, COEUS_KV_F16>(strip, lane, e, row0, col0, em, en);
        } else if (e.kv_dtype == COEUS_KV_BF16) {
            if (e.bias) k64_strip_kv<true, COEUS_KV_BF16>(strip, lane, e, row0, col0, em, en);
            else k64_strip_kv<false, COEUS_KV_BF16>(strip, lane, e, row0, col0, em, en);
        } else {
            if (e.bias) k64_strip_kv<true, COEUS_KV_F32>(strip, lane, e, row0, col0, em, en);
            else k64_strip_kv<false, COEUS_KV_F32>(strip, lane, e, row0, col0, em, en);
        }
    } else if (kind == K64_GATED) {
        const bool clamp = e.act == COEUS_EPI_CLAMP_GATE;
        if (!e.out_lp) {
            if (clamp) k64_strip_gated<true, false>(strip, lane, e, row0, col0, em);
            else k64_strip_gated<false, false>(strip, lane, e, row0, col0, em);
        } else if (e.lp_bf16) {
            if (clamp) k64_strip_gated<true, true, true>(strip, lane, e, row0, col0, em);
            else k64_strip_gated<false, true, true>(strip, lane, e, row0, col0, em);
        } else {
            if (clamp) k64_strip_gated<true, true, false>(strip, lane, e, row0, col0, em);
            else k64_strip_gated<false, true, false>(strip, lane, e, row0, col0, em);
        }
    } else {
        k64_strip_generic(strip, lane, e, gated, vec4, row0, col0, em, en);
    }
}

template <bool BF16>
__global__ __launch_bounds__(256) void gemm_h256k64_kernel(const uint16_t *a, const uint16_t *w, uint64_t m,
                                                           uint64_t n, uint64_t k, uint64_t lda,
                                                           uint64_t ldw, uint32_t tiles_m, uint32_t tiles_n,
                                                           uint32_t splits, uint32_t full_tiles,
                                                           float *tail_part, EpiArgs e) {
    extern __shared__ __attribute__((aligned(16))) uint16_t sm[];  // A regions 0-2, W regions 0-1
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the three kinds of launch of gemm_h256_kernel
    const uint32_t total = tiles_m * tiles_n;
    uint32_t split = 0, bid = blockIdx.x, shares = 1, tail_idx = 0;
    bool tail_wg = false;
    if (tail_part) {
        if (bid >= full_tiles) {
            const uint32_t tail = total - full_tiles, o = bid - full_tiles;
            split = o / tail;
            tail_idx = o - split * tail;
            bid = full_tiles + tail_idx;
            shares = splits;
            tail_wg = true;
        }
    } else if (splits > 1) {
        split = bid / total;
        bid -= split * total;
        shares = splits;
        e.out_f32 += (uint64_t)split * m * e.n_eff;
    }
    const uint64_t nslices = k / UK;
    const uint64_t kbeg = nslices * split / shares * UK, kend = nslices * (split + 1) / shares * UK;
    uint32_t tm, tn;
    h256_tile_of(bid, tiles_m, tiles_n, tm, tn);
    const uint64_t m0 = (uint64_t)tm * TM, n0 = (uint64_t)tn * TN;
    const uint32_t wm = (wave >> 1) * 128, wn = (wave & 1) * 128;
    float16_t acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int y = 0; y < 4; y++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[x][y][i] = 0.f;

    K64Source src;
    src.a = (const char *)(a + m0 * lda);
    src.w = (const char *)(w + n0 * ldw);
    {
        const uint32_t amax = (uint32_t)min((uint64_t)TM - 1, m - 1 - m0), wmax = (uint32_t)min((uint64_t)TN - 1, n - 1 - n0);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            // row = 8 (4 q + wave) + lane / 8; slot lane % 8 holds piece slot ^ (row / 2 % 8)
            const uint32_t row = 8 * (4 * q + wave) + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
            src.oa[q] = min(row, amax) * ((uint32_t)lda * 2) + piece * 16;
            src.ow[q] = min(row, wmax) * ((uint32_t)ldw * 2) + piece * 16;
        }
    }
    K64Lane ln;
    {
        const uint32_t frow = lane & 31, fhf = lane >> 5, fsw = (lane >> 1) & 7;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            ln.a[j] = (wm + frow) * UK + 8 * ((2 * j + fhf) ^ fsw);
            ln.w[j] = (wn + frow) * UK + 8 * ((2 * j + fhf) ^ fsw);
        }
    }
    uint16_t *const rega = sm, *const regw = sm + 3 * UREG;
    auto request_all = [&](uint16_t *region, bool is_w, uint64_t k0) {
#pragma unroll
        for (int q = 0; q < 8; q++) k64_request(src, q, is_w, k0, region, wave);
    };
    // slices past the end are requested as repeats of the last one (and never used), so that the
    // number of loads in flight at each wait does not depend on the number of slices
    const uint64_t klast = kend - UK;
    auto kof = [&](uint64_t j) { return kbeg + j * UK <= klast ? kbeg + j * UK : klast; };
    request_all(rega, false, kbeg);
    request_all(regw, true, kbeg);
    request_all(rega + UREG, false, kof(1));
    request_all(regw + UREG, true, kof(1));
    request_all(rega + 2 * UREG, false, kof(2));
    __builtin_amdgcn_s_waitcnt(0x4F78);  // vmcnt(24): slice 0 has landed (this wave's part)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    K64Frags f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        f.a[0][j] = k64_read(rega, ln.a[j], 0);
#pragma unroll
        for (int y = 0; y < 4; y++) f.b[y][j] = k64_read(regw, ln.w[j], y);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    // slice 0, steps 0-2; W of slice 2 goes where W of slice 0 was
    const uint64_t nsl = (kend - kbeg) / UK;
    k64_period<BF16, true, true>(rega, regw, nullptr, regw, ln, wave, src, kof(2), f, acc);
    // periods s = 0 .. nsl - 2: the last step of slice s and steps 0-2 of slice s + 1
    uint32_t ra = 0, rw = 0;  // regions of slice s
    uint64_t s = 0;
    for (; s + 3 < nsl; s++) {
        const uint32_t ra1 = ra == 2 ? 0 : ra + 1;
        k64_period<BF16, false, true>(rega + ra1 * UREG, regw + (rw ^ 1) * UREG, rega + ra * UREG,
                                      regw + (rw ^ 1) * UREG, ln, wave, src, kbeg + (s + 3) * UK, f, acc);
        ra = ra1;
        rw ^= 1;
    }
    for (; s + 1 < nsl; s++) {
        const uint32_t ra1 = ra == 2 ? 0 : ra + 1;
        k64_period<BF16, false, false>(rega + ra1 * UREG, regw + (rw ^ 1) * UREG, nullptr, nullptr, ln, wave, src, 0,
                                       f, acc);
        ra = ra1;
        rw ^= 1;
    }
    // the last step of the last slice
#pragma unroll
    for (int i = 0; i < 16; i++) mfma_32x32x16<BF16>(f.b[i & 3][i >> 2], f.a[1][i >> 2], acc[3][i & 3]);
    __builtin_amdgcn_s_waitcnt(0x0070);

    // Epilogue through LDS (free now), one 32-row strip of the wave's 128x128 block at a time.
    float *strip = (float *)sm + wave * (32 * 132);
    uint64_t em = m, en = n, em0 = m0, en0 = n0;
    if (tail_wg) {
        EpiArgs pe = {};
        pe.out_f32 = tail_part + ((uint64_t)split * (total - full_tiles) + tail_idx) * (TM * TN);
        pe.n = pe.n_eff = TN;
        pe.vec4 = 1;
        e = pe;
        em = TM; en = TN; em0 = 0; en0 = 0;
    }
    const bool gated = epi_gated(e.act);
    const bool vec4 = e.vec4;
    uint32_t bits;
    const uint32_t kind = k64_epilogue_kind(e, vec4, en0 + wn, en, bits);
    __syncthreads();  // every wave has finished reading the operand slices
    if (kind == K64_GATED && e.out_lp && (e.lp_ld & 7) == 0 && ((uintptr_t)e.out_lp & 15) == 0) {  // 16-byte stores
        const bool clamp = e.act == COEUS_EPI_CLAMP_GATE;
#pragma unroll 1
        for (uint32_t x = 0; x < 4; x++) {
            float16_t t[4];
#define COEUS_T(X) { t[0] = acc[X][0]; t[1] = acc[X][1]; t[2] = acc[X][2]; t[3] = acc[X][3]; }
            if (x == 0) COEUS_T(0)
            else if (x == 1) COEUS_T(1)
            else if (x == 2) COEUS_T(2)
            else COEUS_T(3)
#undef COEUS_T
            const uint64_t row = em0 + wm + x * 32 + (lane & 31);
            if (e.lp_bf16) {
                if (clamp) k64_direct_gated<true, true>(t, lane, e, row, en0 + wn, em);
                else k64_direct_gated<false, true>(t, lane, e, row, en0 + wn, em);
            } else {
                if (clamp) k64_direct_gated<true, false>(t, lane, e, row, en0 + wn, em);
                else k64_direct_gated<false, false>(t, lane, e, row, en0 + wn, em);
            }
        }
        return;
    }
    if (kind == K64_ROWS && (bits & ~1u) == 2) {
        if (bits & 1) k64_epilogue_residual<true>(strip, acc, lane, e, em0 + wm, en0 + wn, em);
        else k64_epilogue_residual<false>(strip, acc, lane, e, em0 + wm, en0 + wn, em);
        return;
    }
    // one copy of the walks for the four row blocks; the accumulators are named with constant
    // indices (indexed dynamically they would live in scratch memory)
#pragma unroll 1
    for (uint32_t x = 0; x < 4; x++) {
        if (x == 0) k64_strip_write(strip, acc[0], lane);
        else if (x == 1) k64_strip_write(strip, acc[1], lane);
        else if (x == 2) k64_strip_write(strip, acc[2], lane);
        else k64_strip_write(strip, acc[3], lane);
        k64_strip_out(strip, lane, e, kind, bits, gated, vec4, em0 + wm + x * 32, en0 + wn, em, en);
    }
}

// ---------------------------------------------------------------- few rows
// Prompts whose 256x256 tiles do not fill the chip leave CUs without work, or split k so often that the planes cost more than the
// products.  So smaller tiles (256 or 128 rows, 64 - 128 columns): eight waves, of which waves 0 - 3 multiply the first two
// 16-wide k steps of every 64-wide slice and waves 4 - 7 the last two (two waves a SIMD, one's fragment reads behind the other's
// products); wave % 4 has RB x NB blocks of 32 x 32, WM rows of waves by 4 / WM.  The two halves are added through LDS.
// Bound by the path from L2 into LDS, which gives a CU 60 - 70 GB/s and all of them 14 - 17 TB/s: 128 (rows + columns) bytes a slice,
// 0.34 us for 128x64 and 0.63 us for 256x96, where the products take 0.12 and 0.36.  The weights come from memory and a slice is
// shorter than that trip: their ring in LDS is deeper than the activations', and waves 0 - 3 request the A rows, waves 4 - 7 the W
// rows, so that neither waits for the other's (a wave's loads return in order).  Layout of a slice as in gemm_h256k64_kernel.
// With all of a slice's fragments read before its products instead of one step ahead: 4096 x 22016 on 201 rows 73.8 us, 59.8 so.
template <int WM, int RB, int NB>
struct NarrowTile {
    static constexpr int WN = 4 / WM, ROWS = WM * RB * 32, COLS = WN * NB * 32;
    static constexpr int UA = ROWS / 32, UW = COLS / 32;  // requests of a wave and slice: 8 rows x 128 bytes each, four waves an operand
    static constexpr int DA = ROWS == 256 ? 3 : 5, DW = ROWS == 256 ? (COLS == 128 ? 4 : COLS == 96 ? 5 : 6) : COLS == 128 ? 5 : 6;
    static constexpr size_t ring = ((size_t)DA * ROWS + (size_t)DW * COLS) * UK * 2, tile = (size_t)ROWS * (COLS + 4) * 4, lds = ring > tile ? ring : tile;
    static_assert(lds <= 160 * 1024, "fits the LDS of a CU");
};

__host__ __device__ constexpr int wait_vm_lds(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0070; }  // vmcnt(n) lgkmcnt(0)

// Requests [Q0, Q1) of a slice: 8 rows x 128 bytes each into LDS.
template <int Q0, int Q1, int Q>
__device__ __forceinline__ void narrow_request(const char *src, const uint32_t (&off)[Q], uint16_t *dst, uint32_t w4) {
    typedef const __attribute__((address_space(1))) void *gptr_t;
    typedef __attribute__((address_space(3))) void *lptr_t;
#pragma unroll
    for (int q = Q0; q < Q1; q++)
        __builtin_amdgcn_global_load_lds((gptr_t)(src + off[q]), (lptr_t)(dst + (4 * q + w4) * 512), 16, 0, 0);
}
// Half a slice: the products of one k step on fragments already in registers, the reads of the next step's fragments between
// them, and requests for a later slice in front (the W rows and the first half of the A rows; SECOND: the other half).  The regions read and the one written
// are distinct (see k64_period).
template <bool BF16, class T, int RB, int NB, bool SECOND, int Q>
__device__ __forceinline__ void narrow_step(const uint16_t *__restrict__ ra, const uint16_t *__restrict__ rw, uint16_t *__restrict__ dst,
                                            const char *src, const uint32_t (&off)[Q], bool takes_a, uint32_t w4, uint32_t la, uint32_t lw,
                                            const uint4 (&af)[RB], const uint4 (&wf)[NB], uint4 (&an)[RB], uint4 (&wn)[NB],
                                            float16_t (&acc)[RB][NB]) {
    if (takes_a) narrow_request<SECOND ? T::UA / 2 : 0, SECOND ? T::UA : T::UA / 2>(src, off, dst, w4);
    else if (!SECOND) narrow_request<0, T::UW>(src, off, dst, w4);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < (RB * NB > RB + NB ? RB * NB : RB + NB); i++) {
        if (i < RB * NB) mfma_32x32x16<BF16>(wf[i / RB], af[i % RB], acc[i % RB][i / RB]);
        if (i < RB) an[i] = k64_read(ra, la, i);
        else if (i < RB + NB) wn[i - RB] = k64_read(rw, lw, i - RB);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// AGAIN: sums begin again every `period` slices, see GemmPlan (a wave of eight blocks has no registers for that).
template <bool BF16, int WM, int RB, int NB, bool AGAIN>
__global__ __launch_bounds__(512) void gemm_narrow_kernel(const uint16_t *a, const uint16_t *w, uint64_t m, uint64_t n, uint64_t k, uint64_t lda,
                                                          uint64_t ldw, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits, uint32_t period, EpiArgs e) {
    using T = NarrowTile<WM, RB, NB>;
    constexpr int DA = T::DA, DW = T::DW, Q = T::UA > T::UW ? T::UA : T::UW;
    constexpr uint32_t RA = T::ROWS * UK, RW = T::COLS * UK;  // elements of a region
    extern __shared__ __attribute__((aligned(16))) uint16_t sm[];  // A regions 0 .. DA - 1, W regions 0 .. DW - 1
    // Workgroups go round-robin to the 8 XCDs: each takes consecutive tiles, rows first, so that its L2 fetches a column tile's
    // weights once (the grid is a multiple of 8).
    const uint32_t tiles = tiles_m * tiles_n, id = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
    if (id >= tiles * splits) return;
    const uint32_t split = id / tiles, r = id - split * tiles, tn = r / tiles_m, tm = r - tn * tiles_m;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), w4 = wave & 3, half = wave >> 2;
    const uint32_t wrow = w4 / T::WN * RB * 32, wcol = w4 % T::WN * NB * 32;
    const uint64_t m0 = (uint64_t)tm * T::ROWS, n0 = (uint64_t)tn * T::COLS;
    const uint64_t nslices = k / UK, kbeg = nslices * split / splits * UK, kend = nslices * (split + 1) / splits * UK;
    if (splits > 1) e.out_f32 += (uint64_t)split * m * e.n_eff;
    float16_t acc[RB][NB];
#pragma unroll
    for (int x = 0; x < RB; x++)
#pragma unroll
        for (int y = 0; y < NB; y++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[x][y][i] = 0.f;
    float16_t total[AGAIN ? RB : 1][AGAIN ? NB : 1];  // of the slices before the present ones
#pragma unroll
    for (int x = 0; x < (AGAIN ? RB : 1); x++)
#pragma unroll
        for (int y = 0; y < (AGAIN ? NB : 1); y++) total[x][y] = acc[x][y];
    const bool takes_a = half == 0;
    uint32_t off[Q];
    {
        const uint32_t last = (uint32_t)(takes_a ? min((uint64_t)T::ROWS - 1, m - 1 - m0) : min((uint64_t)T::COLS - 1, n - 1 - n0));
        const uint32_t ld = (uint32_t)(takes_a ? lda : ldw) * 2;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const uint32_t row = 8 * (4 * q + w4) + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
            off[q] = min(row, last) * ld + piece * 16;
        }
    }
    const char *origin = takes_a ? (const char *)(a + m0 * lda) : (const char *)(w + n0 * ldw);
    // slices past the end are requested as repeats of the last one (and never used): the number of loads in flight at each
    // wait does not depend on the number of slices
    const uint64_t klast = kend - UK;
    auto source = [&](uint64_t kk) { return origin + 2 * (kk < klast ? kk : klast); };
    uint32_t la[2], lw[2];
    {
        const uint32_t frow = lane & 31, fhf = lane >> 5, fsw = (lane >> 1) & 7;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t slot = 8 * ((2 * (2 * half + j) + fhf) ^ fsw);
            la[j] = (wrow + frow) * UK + slot;
            lw[j] = (wcol + frow) * UK + slot;
        }
    }
    uint16_t *const rega = sm, *const regw = sm + DA * RA;
    uint16_t *const ring = takes_a ? rega : regw;
    const uint32_t depth = takes_a ? DA : DW, rsize = takes_a ? RA : RW;
    for (uint32_t j = 0; j < depth; j++) {
        if (takes_a) narrow_request<0, T::UA>(source(kbeg + (uint64_t)j * UK), off, ring + j * RA, w4);
        else narrow_request<0, T::UW>(source(kbeg + (uint64_t)j * UK), off, ring + j * RW, w4);
    }
    // every wave's loads of the next slice have landed (all but the newest `depth - 2` slices'), and it has read all of the last one
    auto meet = [&](auto more) {
        constexpr int D = decltype(more)::value;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        if (takes_a) __builtin_amdgcn_s_waitcnt(wait_vm_lds((DA - 2 + D) * T::UA));
        else __builtin_amdgcn_s_waitcnt(wait_vm_lds((DW - 2 + D) * T::UW));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_sched_barrier(0);
    };
    uint4 af[2][RB], wf[2][NB];
    meet(std::integral_constant<int, 1>{});  // slice 0
#pragma unroll
    for (int x = 0; x < RB; x++) af[0][x] = k64_read(rega, la[0], x);
#pragma unroll
    for (int y = 0; y < NB; y++) wf[0][y] = k64_read(regw, lw[0], y);
    const uint32_t nsl = (uint32_t)((kend - kbeg) / UK);
    // Slice s: the products of its first step, while the second step's fragments are read; then, when nobody reads the slice any
    // more, those of the second, while the next slice's are read.  Slice s + depth goes into the region of slice s.
    uint32_t ia = 0, iw = 0, io = depth - 1;  // regions of slice s; of slice s - 1, whose second half of requests is left
    uint32_t until = period - 1;  // the slice behind which sums begin again
    for (uint32_t s = 0; s < nsl; s++) {
        if (s) {
            narrow_step<BF16, T, RB, NB, true>(rega + ia * RA, regw + iw * RW, ring + io * rsize, source(kbeg + (uint64_t)(s - 1 + depth) * UK), off,
                                               takes_a, w4, la[1], lw[1], af[0], wf[0], af[1], wf[1], acc);
        } else {
#pragma unroll
            for (int x = 0; x < RB; x++) af[1][x] = k64_read(rega, la[1], x);
#pragma unroll
            for (int y = 0; y < NB; y++) wf[1][y] = k64_read(regw, lw[1], y);
#pragma unroll
            for (int i = 0; i < RB * NB; i++) mfma_32x32x16<BF16>(wf[0][i / RB], af[0][i % RB], acc[i % RB][i / RB]);
        }
        meet(std::integral_constant<int, 0>{});
        uint16_t *const freed = ring + (takes_a ? ia : iw) * rsize;
        ia = ia + 1 == DA ? 0 : ia + 1;
        iw = iw + 1 == DW ? 0 : iw + 1;
        io = io + 1 == depth ? 0 : io + 1;
        narrow_step<BF16, T, RB, NB, false>(rega + ia * RA, regw + iw * RW, freed, source(kbeg + (uint64_t)(s + depth) * UK), off, takes_a, w4,
                                            la[0], lw[0], af[1], wf[1], af[0], wf[0], acc);
        if constexpr (AGAIN) {
            if (s == until) {
                until += period;
#pragma unroll
                for (int x = 0; x < RB; x++)
#pragma unroll
                    for (int y = 0; y < NB; y++)
#pragma unroll
                        for (int i = 0; i < 16; i++) { total[x][y][i] += acc[x][y][i]; acc[x][y][i] = 0.f; }
            }
        }
    }
    if constexpr (AGAIN) {
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int y = 0; y < NB; y++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[x][y][i] += total[x][y][i];
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // the repeats have landed too
    __syncthreads();
    // The two halves meet in a [ROWS][COLS + 4] f32 tile; then every thread finishes four (gated: eight) columns of some rows.
    constexpr uint32_t TS = T::COLS + 4;
    float *tile = (float *)sm;
    float *mine = tile + (wrow + (lane & 31)) * TS + wcol + 4 * (lane >> 5);
    if (half == 0) {
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int y = 0; y < NB; y++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    *(float4 *)(mine + x * 32 * TS + y * 32 + 8 * g) = make_float4(acc[x][y][4 * g], acc[x][y][4 * g + 1], acc[x][y][4 * g + 2], acc[x][y][4 * g + 3]);
    }
    __syncthreads();
    if (half == 1) {
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int y = 0; y < NB; y++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    float4 *p = (float4 *)(mine + x * 32 * TS + y * 32 + 8 * g);
                    const float4 o = *p;
                    *p = make_float4(o.x + acc[x][y][4 * g], o.y + acc[x][y][4 * g + 1], o.z + acc[x][y][4 * g + 2], o.w + acc[x][y][4 * g + 3]);
                }
    }
    __syncthreads();
    const bool vec4 = e.vec4;
    const uint32_t live = (uint32_t)min((uint64_t)T::ROWS, m - m0);
    if (!epi_gated(e.act)) {
        constexpr uint32_t CG = T::COLS / 4, RP = 512 / CG;
        const uint32_t c4 = tid % CG * 4;
        if (tid >= RP * CG || n0 + c4 >= n) return;
        const KvCols kc = epi_kv_cols(e, n0 + c4, n);
        for (uint32_t q = tid / CG; q < live; q += RP) {
            const float4 t = *(const float4 *)(tile + q * TS + c4);
            float v[4] = {t.x, t.y, t.z, t.w};
            epi_row4<true>(e, vec4, kc, m0 + q, n0 + c4, n, v);
        }
    } else {
        constexpr uint32_t CG = T::COLS / 8, RP = 512 / CG;
        const uint32_t c8 = tid % CG * 8;
        if (tid >= RP * CG || n0 + c8 >= n) return;
        for (uint32_t q = tid / CG; q < live; q += RP) {
            const float4 p0 = *(const float4 *)(tile + q * TS + c8), p1 = *(const float4 *)(tile + q * TS + c8 + 4);
            const float gv[4] = {p0.x, p0.z, p1.x, p1.z}, uv[4] = {p0.y, p0.w, p1.y, p1.w};
            epi_row4_gated<true>(e, vec4, m0 + q, (n0 + c8) >> 1, n0 + c8, n, gv, uv);
        }
    }
}

template <bool BF16, int WM, int RB, int NB, bool AGAIN = false>
static int launch_narrow(const uint16_t *a, const uint16_t *w, uint64_t m, uint64_t n, uint64_t k, uint64_t lda, uint64_t ldw, uint32_t splits,
                         uint32_t period, const EpiArgs &e, hipStream_t st) {
    if constexpr (!AGAIN && RB * NB < 8)
        if (period != ~0u) return launch_narrow<BF16, WM, RB, NB, true>(a, w, m, n, k, lda, ldw, splits, period, e, st);
    using T = NarrowTile<WM, RB, NB>;
    static const hipError_t once = hipFuncSetAttribute((const void *)gemm_narrow_kernel<BF16, WM, RB, NB, AGAIN>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    COEUS_HIP(once);
    const uint32_t tiles_m = (uint32_t)ceil_div(m, T::ROWS), tiles_n = (uint32_t)ceil_div(n, T::COLS);
    hipLaunchKernelGGL((gemm_narrow_kernel<BF16, WM, RB, NB, AGAIN>), dim3((uint32_t)round_up((uint64_t)tiles_m * tiles_n * splits, 8)), dim3(512), T::lds, st, a, w, m, n,
                       k, lda, ldw, tiles_m, tiles_n, splits, period, e);
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}
template <bool BF16>
static int launch_narrow_plan(uint32_t rows, uint32_t cols, const uint16_t *a, const uint16_t *wp, uint64_t m, const Weight &w, uint64_t lda,
                              uint64_t ldw, uint32_t splits, uint32_t period, const EpiArgs &e, hipStream_t st) {
    if (rows == 256) return cols == 128 ? launch_narrow<BF16, 2, 4, 2>(a, wp, m, w.n, w.k, lda, ldw, splits, period, e, st) : launch_narrow<BF16, 4, 2, 3>(a, wp, m, w.n, w.k, lda, ldw, splits, period, e, st);
    if (cols == 128) return launch_narrow<BF16, 2, 2, 2>(a, wp, m, w.n, w.k, lda, ldw, splits, period, e, st);
    return cols == 96 ? launch_narrow<BF16, 4, 1, 3>(a, wp, m, w.n, w.k, lda, ldw, splits, period, e, st) : launch_narrow<BF16, 4, 1, 2>(a, wp, m, w.n, w.k, lda, ldw, splits, period, e, st);
}


// ---------------------------------------------------------------- f32 weights
// k % 4 == 0: slices of 32 L floats a row (L lines of 128 bytes, laid out like the 64-wide slices of the 16-bit kernels) straight into a ring of D
// regions, two of them on their way while one is multiplied by v_mfma_f32_32x32x2_f32.  A reduction index is only a label: a lane's 16 bytes of a row
// are four k, and instruction i of four sums over the i-th of lanes 0 - 31 and the i-th of lanes 32 - 63.  WM x WN x KH waves: wave (m, n, h) has
// RB x NB blocks of 32 x 32 and multiplies steps h, h + KH ... of a slice's 4 L steps of 8 k; the KH sums of an output meet in LDS.
// A chain of f32 sums is no longer than the 4 L / KH steps of PERIOD slices: their sums are added to those of the slices before.
// Bound: up to some 128 rows by the way of the first slices from memory and the chain of a workgroup's products (6 slices of 768 k, 0.43 us each where
// eight waves share a 32x32 tile), beyond that by the products (157 TF at most).  The kernels before took operands through registers into k-major tiles, with
// 32-byte requests and all requests waited for at each slice.  us, before / this: 768 x 2304, 768 x 768, 768 x 3072, 3072 x 768
//   17 rows    9.4 / 8.1   9.2 / 7.9   9.2 / 7.9   10.8 / 10.2
//   128 rows  12.9 / 11.0  9.4 / 8.2  12.9 / 11.1  19.8 / 15.5
//   512 rows  40.8 / 26.9 13.1 / 11.1 41.1 / 27.1  43.4 / 31.1
//   1024 rows 56.7 / 41.8 22.2 / 18.5 59.6 / 45.5  74.8 / 49.5
// and 4096 x 4096 x 4096 1329 / 1075 (128 TF); 768 x 50257 with 17, 128, 1024 rows 75 / 37, 122 / 101, 805 / 682.
template <int WM, int WN, int RB, int NB, int KH, int L, int D, int PERIOD>
struct F32Tile {
    static constexpr int WAVES = WM * WN * KH, ROWS = WM * RB * 32, COLS = WN * NB * 32, SK = 32 * L, STEPS = 4 * L / KH;
    static constexpr int QA = ROWS / 8 * L / WAVES, QW = COLS / 8 * L / WAVES;  // requests of a wave and slice, 8 rows x 128 bytes each
    static_assert(QA * WAVES * 8 == ROWS * L && QW * WAVES * 8 == COLS * L && STEPS * KH == 4 * L && D >= 2, "whole requests and steps a wave");
    static constexpr size_t region = (size_t)(ROWS + COLS) * L * 128, sums = (size_t)KH * ROWS * (COLS + 4) * 4, lds = D * region > sums ? D * region : sums;
    static_assert(lds <= 160 * 1024, "fits the LDS of a CU");
};

template <int WM, int WN, int RB, int NB, int KH, int L, int D, int PERIOD>
__device__ __forceinline__ void gemm_f32_tile(const float *a, const float *w, uint64_t m, uint64_t n, uint32_t k, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits,
                                              EpiArgs &e) {
    using T = F32Tile<WM, WN, RB, NB, KH, L, D, PERIOD>;
    extern __shared__ __attribute__((aligned(16))) char f32_sm[];
    // consecutive tiles, rows first, on one XCD (see gemm_narrow_kernel; the grid is a multiple of 8)
    const uint32_t tiles = tiles_m * tiles_n, id = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
    if (id >= tiles * splits) return;
    const uint32_t split = id / tiles, r = id - split * tiles, tn = r / tiles_m, tm = r - tn * tiles_m;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), part = wave % KH, wrow = wave / KH / WN * RB * 32, wcol = wave / KH % WN * NB * 32;
    const uint64_t m0 = (uint64_t)tm * T::ROWS, n0 = (uint64_t)tn * T::COLS;
    const uint32_t slices = (k + T::SK - 1) / T::SK, sbeg = (uint32_t)((uint64_t)slices * split / splits), send = (uint32_t)((uint64_t)slices * (split + 1) / splits);
    if (splits > 1) e.out_f32 += (uint64_t)split * m * e.n_eff;
    // what this lane requests: bytes of its rows from the tile's first, and its four k of a slice
    uint32_t row_at[T::QA + T::QW], col_at[T::QA + T::QW];
    {
        const uint32_t last_a = (uint32_t)min((uint64_t)T::ROWS - 1, m - 1 - m0), last_w = (uint32_t)min((uint64_t)T::COLS - 1, n - 1 - n0);
#pragma unroll
        for (int q = 0; q < T::QA + T::QW; q++) {
            const bool is_a = q < T::QA;
            const uint32_t unit = (is_a ? q : q - T::QA) * T::WAVES + wave, per = (is_a ? T::ROWS : T::COLS) / 8;
            const uint32_t row = unit % per * 8 + (lane >> 3);
            row_at[q] = min(row, is_a ? last_a : last_w) * (k * 4);
            col_at[q] = unit / per * 32 + 4 * ((lane & 7) ^ ((row >> 1) & 7));
        }
    }
    const char *const a0 = (const char *)(a + m0 * k), *const w0 = (const char *)(w + n0 * k);
    auto request = [&](uint32_t s, char *region) {  // (behind the end of a row its last four again, behind the last slice that one)
        typedef const __attribute__((address_space(1))) void *gptr_t;
        typedef __attribute__((address_space(3))) void *lptr_t;
        const uint32_t kk = min(s, send - 1) * T::SK;
#pragma unroll
        for (int q = 0; q < T::QA + T::QW; q++) {
            const bool is_a = q < T::QA;
            char *to = region + ((is_a ? q : q - T::QA) * T::WAVES + wave) * 1024 + (is_a ? 0 : T::ROWS * L * 128);
            __builtin_amdgcn_global_load_lds((gptr_t)((is_a ? a0 : w0) + (row_at[q] + 4 * min(kk + col_at[q], k - 4))), (lptr_t)to, 16, 0, 0);
        }
    };
    float16_t acc[RB][NB], total[RB][NB];
#pragma unroll
    for (int x = 0; x < RB; x++)
#pragma unroll
        for (int y = 0; y < NB; y++)
#pragma unroll
            for (int i = 0; i < 16; i++) { acc[x][y][i] = 0.f; total[x][y][i] = 0.f; }
    const uint32_t frow = lane & 31, fsw = (lane >> 1) & 7;
    // the products of a slice; EDGE: k ends inside it (what lies behind takes part as zeros)
    auto multiply = [&](const char *__restrict__ region, uint32_t kk, auto edge) {
        constexpr bool EDGE = decltype(edge)::value;
#pragma unroll
        for (int t = 0; t < T::STEPS; t++) {
            const uint32_t step = t * KH + part, line = step >> 2, piece = 2 * (step & 3) + (lane >> 5);
            const uint32_t at = frow * 128 + 16 * (piece ^ fsw);
            float4_t af[RB], wf[NB];
#pragma unroll
            for (int x = 0; x < RB; x++) af[x] = *(const float4_t *)(region + (line * T::ROWS + wrow + 32 * x) * 128 + at);
#pragma unroll
            for (int y = 0; y < NB; y++) wf[y] = *(const float4_t *)(region + (T::ROWS * L + line * T::COLS + wcol + 32 * y) * 128 + at);
            if (EDGE && kk + 32 * line + 4 * piece >= k) {
#pragma unroll
                for (int x = 0; x < RB; x++) af[x] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int y = 0; y < NB; y++) wf[y] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int x = 0; x < RB; x++)
#pragma unroll
                    for (int y = 0; y < NB; y++) acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[y][i], af[x][i], acc[x][y], 0, 0, 0);
        }
    };
#pragma unroll
    for (int d = 0; d < D - 1; d++) request(sbeg + d, f32_sm + d * T::region);
    // (fetched here: behind the products their trip takes 0.5 us of 11)
    const uint32_t act = e.act, vec4 = e.vec4;
    asm volatile("" ::"s"(act), "s"(vec4));
    uint32_t at = 0, until = PERIOD;
    for (uint32_t s = sbeg; s < send; s++) {
        // every wave's requests of slice s have landed (all but the D - 2 newest slices'), and it has read all of slice s - 1
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(wait_vm_lds((D - 2) * (T::QA + T::QW)));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t before = at == 0 ? D - 1 : at - 1;
        request(s + D - 1, f32_sm + before * T::region);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t kk = s * T::SK;
        if (kk + T::SK <= k) multiply(f32_sm + at * T::region, kk, std::false_type{});
        else multiply(f32_sm + at * T::region, kk, std::true_type{});
        at = at + 1 == D ? 0 : at + 1;
        if (--until == 0) {
            until = PERIOD;
#pragma unroll
            for (int x = 0; x < RB; x++)
#pragma unroll
                for (int y = 0; y < NB; y++)
#pragma unroll
                    for (int i = 0; i < 16; i++) { total[x][y][i] += acc[x][y][i]; acc[x][y][i] = 0.f; }
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // the repeats have landed too
    __syncthreads();
    constexpr uint32_t TS = T::COLS + 4;
    float *sums = (float *)f32_sm;
    {
        float *mine = sums + (part * T::ROWS + wrow + frow) * TS + wcol + 4 * (lane >> 5);
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int y = 0; y < NB; y++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float16_t &c = acc[x][y], &o = total[x][y];
                    *(float4 *)(mine + x * 32 * TS + y * 32 + 8 * g) = make_float4(o[4 * g] + c[4 * g], o[4 * g + 1] + c[4 * g + 1], o[4 * g + 2] + c[4 * g + 2], o[4 * g + 3] + c[4 * g + 3]);
                }
    }
    __syncthreads();
    const uint32_t live = (uint32_t)min((uint64_t)T::ROWS, m - m0);
    auto gather = [&](uint32_t q, uint32_t c4) {
        const float *p = sums + q * TS + c4;
        float4 v = *(const float4 *)p;
#pragma unroll
        for (int h = 1; h < KH; h++) {
            const float4 o = *(const float4 *)(p + h * T::ROWS * TS);
            v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
        }
        return v;
    };
    if (!epi_gated(act)) {
        constexpr uint32_t CG = T::COLS / 4, RP = T::WAVES * 64 / CG;
        const uint32_t c4 = tid % CG * 4;
        if (n0 + c4 >= n) return;
        const KvCols kc = epi_kv_cols(e, n0 + c4, n);
        for (uint32_t q = tid / CG; q < live; q += RP) {
            const float4 t = gather(q, c4);
            float v[4] = {t.x, t.y, t.z, t.w};
            epi_row4<true>(e, vec4, kc, m0 + q, n0 + c4, n, v);
        }
    } else {
        constexpr uint32_t CG = T::COLS / 8, RP = T::WAVES * 64 / CG;
        const uint32_t c8 = tid % CG * 8;
        if (n0 + c8 >= n) return;
        for (uint32_t q = tid / CG; q < live; q += RP) {
            const float4 p0 = gather(q, c8), p1 = gather(q, c8 + 4);
            const float gv[4] = {p0.x, p0.z, p1.x, p1.z}, uv[4] = {p0.y, p0.w, p1.y, p1.w};
            epi_row4_gated<true>(e, vec4, m0 + q, (n0 + c8) >> 1, n0 + c8, n, gv, uv);
        }
    }
}

template <int WM, int WN, int RB, int NB, int KH, int L, int D, int PERIOD>
__global__ __launch_bounds__(WM *WN *KH * 64) void gemm_f32_small_kernel(const float *a, const float *w, uint64_t m, uint64_t n, uint32_t k, uint32_t tiles_m,
                                                                         uint32_t tiles_n, uint32_t splits, EpiArgs e) {
    gemm_f32_tile<WM, WN, RB, NB, KH, L, D, PERIOD>(a, w, m, n, k, tiles_m, tiles_n, splits, e);
}
template <int WM, int WN, int RB, int NB, int KH, int L, int D, int PERIOD>
__global__ __launch_bounds__(WM *WN *KH * 64) void gemm_f32_kernel(const float *a, const float *w, uint64_t m, uint64_t n, uint32_t k, uint32_t tiles_m,
                                                                   uint32_t tiles_n, uint32_t splits, EpiArgs e) {
    gemm_f32_tile<WM, WN, RB, NB, KH, L, D, PERIOD>(a, w, m, n, k, tiles_m, tiles_n, splits, e);
}

// The tiles, and what a launch of them takes: us = 3.0 + max(alone k, rounds rate k + fixed), k in thousands of one share and `rounds` of 256 workgroups;
// a split launch's sums cost 3.8 us and 0.35 us for each MB of partial products.  Fitted to 2600 launches (17 to 1024 rows; k 512 to 4096; n 260 to 50257;
// 1 to 12 shares): the tile and split of least estimated time is on average 0.7 % and at most 9 % slower than the best one of 17 tiles timed.  us, best:
//   rows             32x32 k128      32x32 k64       64x32           64x64           128x64
//   128 x 768 x 768  8.2             9.3             10.9            18              -
//   128 x 3072 x 768 15.7 (2 shares) 15.5 (8)        15.1 (4)        16 (8)          -
//   256 x 768 x 2304 21              16.7            18.2            19.0            34
//   1024 x 768 x 2304 62             45.3            41.8            45.4            56
//   256 x 768 x 50257 350            230             206             183             193
//   1024 x 768 x 50257 1470          893             796             823             709
struct F32Shape { uint32_t rows, cols, slice, waves; double rate, fixed, alone; };
static constexpr F32Shape kF32Shapes[] = {{32, 32, 128, 8, 6.9, 0.1, 0.}, {32, 32, 64, 4, 5.7, 0.9, 8.1}, {64, 32, 64, 8, 9.4, 0.9, 10.4},
                                          {64, 64, 32, 8, 17., 2., 21.},  {128, 64, 32, 8, 32., 2.4, 37.7}};
struct F32Plan { uint32_t shape, splits; };
// A launch of that many workgroups of `waves` waves fits a grid's 2^32 threads (it is rounded up to a multiple of 8).
static constexpr bool f32_grid_fits(uint64_t workgroups, uint32_t waves) { return workgroups < (1ull << 32) / (64 * waves) - 8; }
static F32Plan gemm_f32_plan(const Weight &w, uint64_t m, bool may_split) {
    F32Plan best{0, 0};
    double least = 0.;
    for (uint32_t i = 0; i < sizeof(kF32Shapes) / sizeof(kF32Shapes[0]); i++) {
        const F32Shape &t = kF32Shapes[i];
        const uint64_t tiles = ceil_div(m, t.rows) * ceil_div(w.n, t.cols), slices = ceil_div(w.k, t.slice);
        for (uint32_t s : {1u, 2u, 3u, 4u, 6u, 8u}) {
            if ((s > 1 && (!may_split || slices < 2 * s)) || !f32_grid_fits(tiles * s, t.waves)) break;
            const double k = (double)(ceil_div(slices, s) * t.slice) / 1000.;
            const double us = std::max(t.alone * k, (double)ceil_div(tiles * s, 256) * t.rate * k + t.fixed) + (s > 1 ? 3.8 + 1.4e-6 * s * (double)m * (double)w.n : 0.);
            if (best.splits == 0 || us < least) { least = us; best = {i, s}; }
        }
    }
    return best;
}

// 16-byte requests, 32-bit places in a tile, and a grid for the largest tiles at least
static bool gemm_f32_has_tiles(const Weight &w, uint64_t m) {
    const F32Shape &largest = kF32Shapes[sizeof(kF32Shapes) / sizeof(kF32Shapes[0]) - 1];
    return (w.k & 3) == 0 && w.k < (1u << 22) && f32_grid_fits(ceil_div(m, largest.rows) * ceil_div(w.n, largest.cols), largest.waves);
}

template <int WM, int WN, int RB, int NB, int KH, int L, int D, int PERIOD>
static int launch_f32_tile(const Weight &w, const float *a, uint64_t m, uint32_t splits, const EpiArgs &e, hipStream_t st) {
    using T = F32Tile<WM, WN, RB, NB, KH, L, D, PERIOD>;
    void (*kern)(const float *, const float *, uint64_t, uint64_t, uint32_t, uint32_t, uint32_t, uint32_t, EpiArgs);
    if constexpr (T::ROWS == 32) kern = gemm_f32_small_kernel<WM, WN, RB, NB, KH, L, D, PERIOD>;
    else kern = gemm_f32_kernel<WM, WN, RB, NB, KH, L, D, PERIOD>;
    static const hipError_t room = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)T::lds);
    COEUS_HIP(room);
    const uint32_t tiles_m = (uint32_t)ceil_div(m, T::ROWS), tiles_n = (uint32_t)ceil_div(w.n, T::COLS);
    hipLaunchKernelGGL(kern, dim3((uint32_t)round_up((uint64_t)tiles_m * tiles_n * splits, 8)), dim3(T::WAVES * 64), T::lds, st, a, (const float *)w.data, m, w.n,
                       (uint32_t)w.k, tiles_m, tiles_n, splits, e);
    return COEUS_OK;
}

// Any k: 64x64 tiles, or 32x32 where there are fewer of those than CUs.  A long k on few tiles is split: at least 12 slices a share and about three
// workgroups a CU in all (below 48 slices the second launch costs what the split saves).
static bool gemm_f32_any_is_small(const Weight &w, uint64_t m) { return ceil_div(w.n, BN) * ceil_div(m, BM) < 256; }
static uint32_t gemm_f32_any_splits(const Weight &w, uint64_t m) {
    const uint64_t slices = ceil_div(w.k, BK);
    if (m == 0 || !gemm_f32_any_is_small(w, m) || slices < 48) return 1;
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>({768 / (ceil_div(w.n, SN) * ceil_div(m, SM)), slices / 12, 8}));
}
static uint32_t gemm_f32_splits_wanted(const Weight &w, uint64_t m) {
    if (m == 0 || gemv_takes_f32_rows(w, m)) return 1;
    return gemm_f32_has_tiles(w, m) ? gemm_f32_plan(w, m, true).splits : gemm_f32_any_splits(w, m);
}

static int launch_gemm_f32(const Weight &w, const float *a, uint64_t m, const Epilogue &ep,
                           const GemmScratch &scr, hipStream_t st) {
    // Up to 16 rows: the decode matmul, which gives a weight row's k to 16 waves and requests all of it at once (768 x 2304 / 768 x 768 /
    // 768 x 3072 / 3072 x 768: 16 rows 4.3 / 4.1 / 4.4 / 9.4 us there, 17 rows 8.1 / 7.9 / 7.9 / 10.2 us here).
    if (gemv_takes_f32_rows(w, m)) {
        if (scr.ev_begin) COEUS_HIP(hipEventRecord(scr.ev_begin, st));
        for (uint32_t rep = 0; rep < (scr.repeat ? scr.repeat : 1); rep++) COEUS_TRY(launch_gemv(w, a, m, ep, st));
        if (scr.ev_end) COEUS_HIP(hipEventRecord(scr.ev_end, st));
        return COEUS_OK;
    }
    const EpiArgs e = make_epi(ep, w.n);
    const bool tiled = gemm_f32_has_tiles(w, m) && ((uintptr_t)a & 15) == 0, small = gemm_f32_any_is_small(w, m);
    F32Plan plan{0, 1};
    for (bool may : {true, false}) {
        plan = tiled ? gemm_f32_plan(w, m, may) : F32Plan{0, may ? gemm_f32_any_splits(w, m) : 1};
        if (plan.splits == 1 || (scr.partials && scr.partials_bytes >= (uint64_t)plan.splits * m * w.n * 4)) break;
    }
    const uint32_t splits = plan.splits;
    EpiArgs plain;  // a split launch stores bare products: [split][m][n] f32
    if (splits > 1) {
        Epilogue pe;
        pe.out_f32 = scr.partials;
        plain = make_epi(pe, w.n);
    }
    const EpiArgs &ke = splits > 1 ? plain : e;
    const uint64_t groups = ceil_div(w.n, epi_gated(e.act) ? 8 : 4);
    const dim3 any_grid((unsigned)ceil_div(w.n, small ? SN : BN), (unsigned)ceil_div(m, small ? SM : BM), splits);
    if (scr.ev_begin) COEUS_HIP(hipEventRecord(scr.ev_begin, st));
    for (uint32_t rep = 0; rep < (scr.repeat ? scr.repeat : 1); rep++) {
        if (tiled) {
            switch (plan.shape) {
                case 0: COEUS_TRY((launch_f32_tile<1, 1, 1, 1, 8, 4, 3, 2>(w, a, m, splits, ke, st))); break;
                case 1: COEUS_TRY((launch_f32_tile<1, 1, 1, 1, 4, 2, 3, 4>(w, a, m, splits, ke, st))); break;
                case 2: COEUS_TRY((launch_f32_tile<2, 1, 1, 1, 4, 2, 3, 4>(w, a, m, splits, ke, st))); break;
                case 3: COEUS_TRY((launch_f32_tile<2, 2, 1, 1, 2, 1, 3, 4>(w, a, m, splits, ke, st))); break;
                default: COEUS_TRY((launch_f32_tile<4, 2, 1, 1, 1, 1, 3, 2>(w, a, m, splits, ke, st))); break;
            }
        } else if (small) {
            auto kern = ke.kv_k ? gemm_f32_any_small_kernel<true> : gemm_f32_any_small_kernel<false>;
            hipLaunchKernelGGL(kern, any_grid, dim3(256), 0, st, a, (const float *)w.data, m, w.n, w.k, splits, ke);
        } else {
            auto kern = ke.kv_k ? gemm_f32_any_kernel<true> : gemm_f32_any_kernel<false>;
            hipLaunchKernelGGL(kern, any_grid, dim3(256), 0, st, a, (const float *)w.data, m, w.n, w.k, ke);
        }
        if (splits > 1)
            hipLaunchKernelGGL(gemm_split_reduce_kernel, dim3((unsigned)ceil_div(m * groups, 256)), dim3(256), 0, st,
                               (const float *)scr.partials, splits, m, w.n, e);
    }
    if (scr.ev_end) COEUS_HIP(hipEventRecord(scr.ev_end, st));
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// Any number of rows: a short prompt leaves most of a 256-row tile empty (rows past the end are
// clamped on the way in and not stored), and is still several times faster here than in the
// 128x128 register-staged kernel (1B shape, 16 rows: 24.5 ms per prompt pass there).
static bool gemm_uses_h256(const Weight &w, uint64_t m) {
    return w.dtype != COEUS_W_F32 && (w.k % TK) == 0 && m >= 1 && w.n >= 128 &&
           (uint64_t)TM * gemm_ld(w.k) < (1ull << 31);  // the byte offsets within a tile fit 32 bits
}

// A launch of few tiles (short prompts, narrow matrices) leaves most CUs without a workgroup while
// each tile walks all of k at about a microsecond per 32-wide slice.  Such launches are split along
// k: `splits` workgroups per tile each take a share of the slices and store plain partial products,
// and a second kernel sums them in split order (deterministic) and runs the epilogue.  At least 8
// slices per split (the request pipeline is 3 deep), at most 16 splits, no more workgroups than CUs (one workgroup
// fills a CU's LDS).  Each split adds a plane of m x n floats to write and read back: of the splits that fit, the one
// with the shortest sum of 0.6 us per slice of the longest share, 4.5 us for the second launch and the planes at 5.5 TB/s (us, the most
// splits that fit / this rule: 201 rows of 4096 x 4096 34.6 / 31.5, of 768 x 3072 22.9 / 22.9; 512 rows of 768 x 3072
// 29.5 / 24.9; 2000 rows of 768 x 2304 35.4 / 28.0).  k % 64 == 0: shares are made of 64-wide slices (counted in 32s, 256 rows of
// 2048 x 3072 got six uneven shares instead of eight even ones, 29.3 against 27.4 us; 700 of 1024 x 2048 three instead of four, 31.1 /
// 29.2).  Over 389 launches of 24 matrices and 65 - 2000 rows, each timed with every number of splits that fits: 0.7 % above the
// fastest one on average (most that fit 2.9 %, counted in 32s 0.9 %), 8 % at worst; 16 of them are 2 - 7 % slower than with the
// most that fit (256 rows of 1536 x 4096 28.4 with six, 30.2 with the four of this rule).
static uint32_t gemm_splits_wanted(const Weight &w, uint64_t m) {
    if (!gemm_uses_h256(w, m)) return 1;
    const uint64_t tiles = ceil_div(m, TM) * ceil_div(w.n, TN), slices = w.k / TK, unit = w.k % UK == 0 ? UK / TK : 1;
    if (tiles > 128) return 1;
    uint64_t most = 256 / tiles;
    if (most > slices / 8) most = slices / 8;
    if (most > 16) most = 16;
    uint32_t best = 1;
    double best_us = 0.6 * (double)slices;
    for (uint64_t s = 2; s <= most; s++) {
        const double us = 0.6 * (double)(ceil_div(slices / unit, s) * unit) + 4.5 + (double)(s * m * w.n) * 8.0 / 5.5e6;
        if (us < best_us) { best_us = us; best = (uint32_t)s; }
    }
    return best;
}

// Which kernel and how many shares of k a launch of k % 64 == 0 takes: rows 0 = the 256x256 tiles.  Launches that fill more than one
// round of those keep them.  Else the estimate below is taken for every narrow tile and number of shares, and the shortest
// one runs if it is under 0.95 of the 256x256 kernel's: per round of 256 workgroups 3.6 us and 0.25 us per 1024 outputs of a
// tile, per slice the tile's 128 (rows + columns) bytes at 66 GB/s a CU and 17 TB/s in all (what the path from L2 into LDS
// gives), for several shares 5.8 us and the planes at 4.4 TB/s; 256x256: 14 us and 0.9 us a slice.  Fitted to 19 matrices of
// 768 - 22016 with 65 - 2036 rows, every tile and number of shares timed: 1 % above the fastest on average, 13 % at worst
// (2048 x 2048, 65 rows, 12.6 against 11.2 us).  us, 256x256 tiles / this: 201 rows of 4096 x 4096 32.8 / 21.7, of 4096 x 12288
// 53.0 / 38.3, of 4096 x 22016 70.8 / 59.8, of 11008 x 4096 56.2 / 39.4; 512 of 768 x 3072 25.3 / 9.4, of 3072 x 768
// 28.3 / 16.3; 1019 of 4096 x 4096 55.6 / 44.4; 2036 of 2048 x 2048 42.6 / 27.5, of 1024 x 2048 30.9 / 17.8.
// Roundings: a result is the end of a chain of k / 16 sums in the 256x256 tiles, of k / 32 here, divided by the shares, and of the
// shares' sum.  Few shares of a long k were up to twice as far from 64 bits as the tiles whose place they take.  So sums begin again every
// `period` slices, as seldom as makes the chain no longer than theirs; 256x128 has no registers for that and is taken where its
// shares are at least half as many.  bf16, root mean square error in 1e-8 of the result's, 256x256 tiles / without that / so, and us without / with:
// 700 rows of 5632 x 2048 15.9 / 32.3 / 15.7, 31.1 / 32.8; 300 of 4096 x 4096 13.7 / 27.1 / 13.3, 25.4 / 25.7; 201 of 4096 x 4096
// 13.6 / 18.8 / 13.3, 20.4 / 20.6; 512 of 768 x 768 9.3 / 11.0 / 8.3, 8.2 / 8.7; 65 of 2048 x 8192 10.2 / 18.5 / 9.8, 14.6 / 15.5.
struct GemmPlan { uint32_t rows = 0, cols = 0, splits = 1, period = ~0u; };
static constexpr uint32_t kNarrowTiles[][2] = {{256, 128}, {256, 96}, {128, 128}, {128, 96}, {128, 64}};
static GemmPlan gemm_plan(const Weight &w, uint64_t m, bool may_split) {
    GemmPlan best;
    best.splits = may_split ? gemm_splits_wanted(w, m) : 1;
    const uint64_t tiles256 = ceil_div(m, TM) * ceil_div(w.n, TN), slices = w.k / UK;
    if (!gemm_uses_h256(w, m) || w.k % UK || tiles256 > 256) return best;
    auto sum_us = [&](uint64_t splits) { return splits > 1 ? 5.8 + (double)(splits * m * w.n) * 8.0 / 4.4e6 : 0.0; };
    const uint64_t shares = best.splits;
    double best_us = 0.95 * (14.0 + 0.9 * (double)ceil_div(slices, shares) + sum_us(shares));
    for (const auto &t : kNarrowTiles) {
        const uint64_t tiles = ceil_div(m, t[0]) * ceil_div(w.n, t[1]);
        for (uint64_t s = 1; s <= (may_split ? 16 : 1) && (s == 1 || (tiles * s <= 256 && slices / s >= 3)); s++) {
            if (t[0] * t[1] == 256 * 128 && 2 * s < shares) continue;
            const double kb = 0.125 * (t[0] + t[1]), busy = (double)std::min<uint64_t>(256, tiles * s);
            const double us = (double)ceil_div(tiles * s, 256) * (3.6 + 0.25 * t[0] * t[1] / 1024.0 + (double)ceil_div(slices, s) * kb * std::max(1 / 66.0, busy / 17e3)) + sum_us(s);
            if (us < best_us) { best_us = us; best.rows = t[0]; best.cols = t[1]; best.splits = (uint32_t)s; }
        }
    }
    if (best.rows && best.rows * best.cols < 256 * 128) {
        auto planes = [](uint64_t s) { return s > 1 ? s : 0; };
        const uint64_t share = ceil_div(slices, best.splits), most = 4 * ceil_div(slices, shares) + planes(shares);
        auto chain = [&](uint64_t parts) { return ceil_div(2 * share, parts) + parts + planes(best.splits); };
        uint64_t parts = 1;
        while (chain(parts) > most && chain(parts + 1) < chain(parts)) parts++;
        if (parts > 1) best.period = (uint32_t)ceil_div(share, parts);
    }
    return best;
}

// A larger launch runs its tiles in rounds of 256 (one workgroup fills a CU), and the last round
// is rarely full: 1376 tiles are five rounds and 96 tiles, which take as long as a sixth round.
// When that remainder is at most half a round its tiles alone are split along k (as many shares
// as fit in one round), through private 256x256 partial tiles and gemm_tail_reduce_kernel.
// Returns the number of shares (1: no split) and the number of tiles of the complete rounds.
static uint32_t gemm_tail_splits_wanted(const Weight &w, uint64_t m, uint32_t *full_tiles) {
    *full_tiles = 0;
    if (!gemm_uses_h256(w, m)) return 1;
    const uint64_t tiles = ceil_div(m, TM) * ceil_div(w.n, TN), slices = w.k / TK;
    const uint64_t full = tiles / 256 * 256, tail = tiles - full;
    if (full == 0 || tail == 0 || tail > 128 || tiles > 0xffffffffull / 16) return 1;
    uint64_t s = 256 / tail;
    if (s > slices / 8) s = slices / 8;
    if (s > 16) s = 16;
    if (s < 2) return 1;
    *full_tiles = (uint32_t)full;
    return (uint32_t)s;
}

uint64_t gemm_split_scratch_bytes(const Weight &w, uint64_t m) {
    if (w.dtype == COEUS_W_F32) {
        const uint32_t sf = gemm_f32_splits_wanted(w, m);
        return sf > 1 ? (uint64_t)sf * m * w.n * 4 : 0;
    }
    if (gemm_uses_few(w, m)) return 0;
    if (gemm_uses_qskinny(w, m)) return gemm_qskinny_scratch_bytes(w, m);
    const GemmPlan plan = gemm_plan(w, m, true);
    if (plan.splits > 1) return (uint64_t)plan.splits * m * w.n * 4;
    if (plan.rows) return 0;
    uint32_t full = 0;
    const uint32_t st = gemm_tail_splits_wanted(w, m, &full);
    if (st > 1) return (uint64_t)st * (ceil_div(m, TM) * ceil_div(w.n, TN) - full) * TM * TN * 4;
    return 0;
}

coeus_matmul_plan gemm_launch_plan(const Weight &w, uint64_t m) {
    if (w.dtype == COEUS_W_F32) {
        if (gemv_takes_f32_rows(w, m)) return gemv_plan(w, m);
        if (!gemm_f32_has_tiles(w, m)) {
            if (gemm_f32_any_is_small(w, m)) return {"gemm_f32_any_small_kernel", SM, SN, 4, gemm_f32_any_splits(w, m), 1};
            return {"gemm_f32_any_kernel", BM, BN, 4, 1, 1};
        }
        const F32Plan plan = gemm_f32_plan(w, m, true);
        const F32Shape &t = kF32Shapes[plan.shape];
        return {t.rows == 32 ? "gemm_f32_small_kernel" : "gemm_f32_kernel", t.rows, t.cols, t.waves, plan.splits, 1};
    }
    if (gemm_uses_few(w, m)) return gemm_few_plan(w, m);
    if (gemm_uses_qskinny(w, m)) return {"gemm_qskinny_kernel", 64, 0, 4, qskinny_splits(w), 1};
    if (!gemm_uses_h256(w, m)) return {"gemm_h_kernel", HM, HN, 4, 1, 1};
    const GemmPlan plan = gemm_plan(w, m, true);
    if (plan.rows) return {"gemm_narrow_kernel", plan.rows, plan.cols, 8, plan.splits, 1};
    uint32_t full = 0;
    const uint32_t tail = plan.splits == 1 ? gemm_tail_splits_wanted(w, m, &full) : 1;
    return {w.k % UK == 0 ? "gemm_h256k64_kernel" : "gemm_h256_kernel", TM, TN, w.k % UK == 0 ? 4u : 8u, plan.splits, tail};
}

bool gemm_appends_kv(const Weight &w, uint64_t m, uint64_t inner, uint64_t hd) {
    // (f32: element by element, or four columns at a time, which stay inside one head)
    if (w.dtype == COEUS_W_F32) return m < (1ull << 32) && w.n == 3 * inner && (inner & 3) == 0 && (hd & 3) == 0;
    if (gemm_uses_few(w, m)) return w.n == 3 * inner;  // (element by element)
    // rows fit 32 bits; a lane's 4 columns stay inside one head.  (The short-prompt kernel for
    // quantised weights qualifies when it is split along k: the kernel that sums its partial
    // planes runs this same epilogue.)
    return gemm_uses_h256(w, m) && (!gemm_uses_qskinny(w, m) || gemm_qskinny_scratch_bytes(w, m) > 0) && m < (1ull << 32) && w.n == 3 * inner && (inner & 3) == 0 && (hd & 3) == 0;
}

int launch_gemm(const Weight &w, const void *a_in, uint64_t m, const Epilogue &ep, GemmScratch &scr,
                hipStream_t st, bool a_staged) {
    const float *a = (const float *)a_in;
    if (m == 0) return fail(COEUS_INVALID_INPUT, "matmul with zero rows");
    if (epi_gated(ep.act) && (w.n & 1))
        return fail(COEUS_INVALID_INPUT, "gated epilogue needs an even number of weight rows");
    if (ep.out_xq) return fail(COEUS_INVALID_INPUT, "prefill matmul has no xq output");
    if (ep.act >= COEUS_EPI_CLAMP_GATE && w.dtype >= COEUS_W_Q8_0)
        return fail(COEUS_INVALID_INPUT, "epilogue %u takes f32 or bf16 weights", ep.act);
    if (w.dtype == COEUS_W_F32) {
        if (a_staged) return fail(COEUS_INVALID_INPUT, "f32 weights take f32 activations");
        return launch_gemm_f32(w, a, m, ep, scr, st);
    }
    const uint64_t lda = gemm_ld(w.k), a_bytes = m * lda * 2;
    const uint16_t *wp = (const uint16_t *)w.data;
    const bool bf = w.dtype == COEUS_W_BF16;
    uint64_t ldw = w.k;
    const uint16_t *ap = (const uint16_t *)a_in;
    if (!a_staged) {
        if (!scr.a_lp || scr.a_lp_bytes < a_bytes)
            return fail(COEUS_INVALID_INPUT, "matmul staging buffer too small (%llu < %llu bytes)",
                        (unsigned long long)scr.a_lp_bytes, (unsigned long long)a_bytes);
        COEUS_TRY(launch_f32_to_16(a, scr.a_lp, m, w.k, lda, bf, st));
        ap = (const uint16_t *)scr.a_lp;
    }
    if (gemm_uses_few(w, m)) {
        const EpiArgs e = make_epi(ep, w.n);
        if (scr.ev_begin) COEUS_HIP(hipEventRecord(scr.ev_begin, st));
        for (uint32_t rep = 0; rep < (scr.repeat ? scr.repeat : 1); rep++) COEUS_TRY(launch_gemm_few(w, ap, lda, m, e, st));
        if (scr.ev_end) COEUS_HIP(hipEventRecord(scr.ev_end, st));
        return COEUS_OK;
    }
    const uint64_t qs_bytes = gemm_uses_qskinny(w, m) ? gemm_qskinny_scratch_bytes(w, m) : 0;
    if (gemm_uses_qskinny(w, m) && (qs_bytes ? scr.partials && scr.partials_bytes >= qs_bytes : !ep.kv_rows_per_seq)) {
        // up to 64 rows on quantised weights: the kernel that streams the quantised blocks
        const EpiArgs e = make_epi(ep, w.n);
        if (scr.ev_begin) COEUS_HIP(hipEventRecord(scr.ev_begin, st));
        for (uint32_t rep = 0; rep < (scr.repeat ? scr.repeat : 1); rep++) {
            uint32_t splits = 1;
            COEUS_TRY(launch_gemm_qskinny(w, ap, lda, m, e, scr.partials, scr.partials_bytes, &splits, st));
            if (splits > 1) {
                const uint64_t groups = ceil_div(w.n, epi_gated(e.act) ? 8 : 4);
                hipLaunchKernelGGL(gemm_split_reduce_kernel, dim3((unsigned)ceil_div(m * groups, 256)), dim3(256), 0, st,
                                   (const float *)scr.partials, splits, m, w.n, e);
            }
        }
        if (scr.ev_end) COEUS_HIP(hipEventRecord(scr.ev_end, st));
        COEUS_HIP(hipGetLastError());
        return COEUS_OK;
    }
    if (!bf) {
        ldw = gemm_ld(w.k);
        const uint64_t w_bytes = w.n * ldw * 2;
        if (!w.expanded) COEUS_TRY(weight_expand(w, scr.expand_budget, st));
        if (w.expanded) {
            wp = (const uint16_t *)w.expanded;
        } else {
            if (!scr.w_lp || scr.w_lp_bytes < w_bytes)
                return fail(COEUS_INVALID_INPUT, "weight staging buffer too small (%llu < %llu bytes)",
                            (unsigned long long)scr.w_lp_bytes, (unsigned long long)w_bytes);
            COEUS_TRY(launch_dequant_to_f16(w, (__half *)scr.w_lp, ldw, st));
            wp = (const uint16_t *)scr.w_lp;
        }
    }
    const EpiArgs e = make_epi(ep, w.n);
    if (ep.kv_rows_per_seq && !gemm_appends_kv(w, m, ep.kv_inner, ep.kv_hd))
        return fail(COEUS_INVALID_INPUT, "this matmul cannot append to the cache (see gemm_appends_kv)");
    if (gemm_uses_h256(w, m)) {
        const size_t lds = (size_t)NSTAGE * (TM + TN) * TK * 2, lds64 = (size_t)5 * UREG * 2;
        static const bool once = [] {
            (void)hipFuncSetAttribute((const void *)gemm_h256_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            (void)hipFuncSetAttribute((const void *)gemm_h256_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            (void)hipFuncSetAttribute((const void *)gemm_h256k64_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            (void)hipFuncSetAttribute((const void *)gemm_h256k64_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            return true;
        }();
        (void)once;
        const uint32_t tiles_m = (uint32_t)ceil_div(m, TM), tiles_n = (uint32_t)ceil_div(w.n, TN);
        // split along k (every tile, or the tiles of the last round) when the caller's scratch has
        // room for the partial products
        GemmPlan plan = gemm_plan(w, m, true);
        if (plan.splits > 1 && (!scr.partials || scr.partials_bytes < (uint64_t)plan.splits * m * w.n * 4)) plan = gemm_plan(w, m, false);
        const uint32_t splits = plan.splits;
        uint32_t full_tiles = 0, tail_splits = 1;
        if (splits == 1 && !plan.rows) {
            tail_splits = gemm_tail_splits_wanted(w, m, &full_tiles);
            if (tail_splits > 1 && (!scr.partials || scr.partials_bytes < gemm_split_scratch_bytes(w, m)))
                tail_splits = 1;
        }
        const uint32_t tail_tiles = tail_splits > 1 ? tiles_m * tiles_n - full_tiles : 0;
        float *tail_part = tail_splits > 1 ? scr.partials : nullptr;
        const dim3 grid(tail_splits > 1 ? full_tiles + tail_tiles * tail_splits : tiles_m * tiles_n * splits);
        const uint32_t ksplits = tail_splits > 1 ? tail_splits : splits;
        EpiArgs plain;  // the split kernels store bare products: [split][m][n] f32
        if (splits > 1) {
            Epilogue pe;
            pe.out_f32 = scr.partials;
            plain = make_epi(pe, w.n);
        }
        const EpiArgs &ke = splits > 1 ? plain : e;
        const uint64_t groups = ceil_div(w.n, epi_gated(e.act) ? 8 : 4);
        if (scr.ev_begin) COEUS_HIP(hipEventRecord(scr.ev_begin, st));
        for (uint32_t rep = 0; rep < (scr.repeat ? scr.repeat : 1); rep++) {
            if (plan.rows)
                COEUS_TRY(bf ? launch_narrow_plan<true>(plan.rows, plan.cols, ap, wp, m, w, lda, ldw, splits, plan.period, ke, st)
                             : launch_narrow_plan<false>(plan.rows, plan.cols, ap, wp, m, w, lda, ldw, splits, plan.period, ke, st));
            else if (w.k % UK == 0 && bf)
                hipLaunchKernelGGL(gemm_h256k64_kernel<true>, grid, dim3(256), lds64, st, ap, wp, m, w.n, w.k, lda, ldw, tiles_m, tiles_n, ksplits, full_tiles, tail_part, ke);
            else if (w.k % UK == 0)
                hipLaunchKernelGGL(gemm_h256k64_kernel<false>, grid, dim3(256), lds64, st, ap, wp, m, w.n, w.k, lda, ldw, tiles_m, tiles_n, ksplits, full_tiles, tail_part, ke);
            else if (bf)
                hipLaunchKernelGGL(gemm_h256_kernel<true>, grid, dim3(512), lds, st, ap, wp, m, w.n, w.k, lda, ldw, tiles_m, tiles_n, ksplits, full_tiles, tail_part, ke);
            else
                hipLaunchKernelGGL(gemm_h256_kernel<false>, grid, dim3(512), lds, st, ap, wp, m, w.n, w.k, lda, ldw, tiles_m, tiles_n, ksplits, full_tiles, tail_part, ke);
            if (splits > 1)
                hipLaunchKernelGGL(gemm_split_reduce_kernel, dim3((unsigned)ceil_div(m * groups, 256)), dim3(256), 0, st,
                                   (const float *)scr.partials, splits, m, w.n, e);
            if (tail_splits > 1)
                hipLaunchKernelGGL(gemm_tail_reduce_kernel, dim3(tail_tiles * 64), dim3(256), 0, st,
                                   (const float *)scr.partials, tail_splits, full_tiles, tiles_m, tiles_n, m, w.n, e);
        }
        if (scr.ev_end) COEUS_HIP(hipEventRecord(scr.ev_end, st));
        COEUS_HIP(hipGetLastError());
        return COEUS_OK;
    }
    const dim3 grid((unsigned)ceil_div(w.n, HN), (unsigned)ceil_div(m, HM));
    if (scr.ev_begin) COEUS_HIP(hipEventRecord(scr.ev_begin, st));
    for (uint32_t rep = 0; rep < (scr.repeat ? scr.repeat : 1); rep++) {
        if (bf)
            hipLaunchKernelGGL(gemm_h_kernel<true>, grid, dim3(256), 0, st, ap, wp, m, w.n, w.k, lda, ldw, e);
        else
            hipLaunchKernelGGL(gemm_h_kernel<false>, grid, dim3(256), 0, st, ap, wp, m, w.n, w.k, lda, ldw, e);
    }
    if (scr.ev_end) COEUS_HIP(hipEventRecord(scr.ev_end, st));
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

}  // namespace coeus
