// Decode matmul: y[b, :] = x[b, :] . W for b < batch <= 16 (math::matmul, MT:50-74, with
// m = batch), the HBM-bound kernel of token generation.
//
//   gemv_quad_kernel   Q8_0 / Q4_0 weights in MFMA-native tiles, batches of 1 and 2 and some of 3 and 4 (the
//                      kernel of single-sequence generation): one workgroup per tile of 16 output rows, a
//                      wave owns four consecutive 128-k chunks, stages exactly their activations
//                      (with or without the folded norm) into its private slice of LDS and feeds
//                      the quants to v_mfma_f32_16x16x32_f16 as f16 subnormals.
//   gemv_rows_kernel   the same weights for batches of 3 to 16 and prompts of up to 16 rows.  One workgroup owns one to six tiles
//                      of 16 output rows; its waves take 128-k chunks (1 KiB of Q4_0 quants = one
//                      fully coalesced 16 B/lane load per wave).  Each 32-k block is one
//                      v_mfma_f32_16x16x32_f16 between the 16 activation rows (f16, straight from
//                      L2 into registers) and the block's integers (q-8 resp. q, exact in f16); the
//                      f32 block result is scaled by the block's f16 scale on the VALU.  In both
//                      kernels the value used for every weight is exactly its dequantised value q*d.
//   gemv_dense_kernel  f32 / bf16 weights, one wave per output row, f32 FMA on the VALU.
//   gemv_row_kernel    one activation row behind a norm of up to 1024 elements: the row in every
//                      wave's registers, no LDS and no barrier.
//   gemv_many_kernel   one plain activation row: two weight rows a wave, up to four steps of both in flight.
//   gemv_mfma_kernel   2 - 16 activation rows on f32 / bf16 weights: 16 output rows a workgroup on
//                      the matrix cores (bf16: the f32 activations as three bf16 each, or prompts'
//                      rows of bf16).
#include "device_utils.hpp"
#include <type_traits>

namespace coeus {

// ---------------------------------------------------------------- xq packing
__global__ void pack_xq_kernel(const float *x, uint32_t batch, uint32_t bp, uint64_t k,
                               uint64_t k_pad, __half *xq) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= k_pad * bp) return;
    const uint32_t e = idx & 7, b = (idx >> 3) % bp;
    const uint64_t kk = (idx >> 3) / bp * 8 + e;
    const float v = (b < batch && kk < k) ? x[(uint64_t)b * k + kk] : 0.0f;
    xq[idx] = __float2half_rn(v);
}

int launch_pack_xq(const float *x, uint64_t batch, uint64_t k, uint64_t k_pad, __half *xq,
                   hipStream_t st) {
    const uint32_t bp = pad_batch(batch);
    hipLaunchKernelGGL(pack_xq_kernel, dim3((unsigned)ceil_div(k_pad * bp, 256)), dim3(256), 0, st,
                       x, (uint32_t)batch, bp, k, k_pad, xq);
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// ---------------------------------------------------------------- quantised kernel
// Q4_0 dword (nibble positions [k0,k2,k4,k6,k1,k3,k5,k7]) -> 8 f16 values q-8, exact:
// 0x6400|n is the f16 1024+n; 0x6400|(n<<4) is 1024+16n, and (1024+16n)/16 - 72 = n - 8.
__device__ __forceinline__ half8_t unpack_q4(uint32_t q) {
    const uint32_t q8 = q >> 8;
    union { uint32_t u; half2_t h; } a, b, c, d;
    a.u = (q & 0x000F000Fu) | 0x64006400u;
    b.u = (q & 0x00F000F0u) | 0x64006400u;
    c.u = (q8 & 0x000F000Fu) | 0x64006400u;
    d.u = (q8 & 0x00F000F0u) | 0x64006400u;
    const half2_t off_lo = {(_Float16)1032.0f, (_Float16)1032.0f};
    const half2_t sc_hi = {(_Float16)0.0625f, (_Float16)0.0625f};
    const half2_t off_hi = {(_Float16)72.0f, (_Float16)72.0f};
    const half2_t r0 = a.h - off_lo, r1 = b.h * sc_hi - off_hi;
    const half2_t r2 = c.h - off_lo, r3 = d.h * sc_hi - off_hi;
    half8_t out = {r0.x, r0.y, r1.x, r1.y, r2.x, r2.y, r3.x, r3.y};
    return out;
}

// Two dwords of int8 -> 8 f16, exact: byte^0x80 = q+128; 0x6400|(q+128) = 1152+q.
__device__ __forceinline__ half8_t unpack_q8(uint32_t lo, uint32_t hi) {
    const uint32_t l = lo ^ 0x80808080u, h = hi ^ 0x80808080u;
    union { uint32_t u; half2_t h2; } a, b, c, d;
    a.u = __builtin_amdgcn_perm(0x64646464u, l, 0x04010400u);
    b.u = __builtin_amdgcn_perm(0x64646464u, l, 0x04030402u);
    c.u = __builtin_amdgcn_perm(0x64646464u, h, 0x04010400u);
    d.u = __builtin_amdgcn_perm(0x64646464u, h, 0x04030402u);
    const half2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const half2_t r0 = a.h2 - off, r1 = b.h2 - off, r2 = c.h2 - off, r3 = d.h2 - off;
    half8_t out = {r0.x, r0.y, r1.x, r1.y, r2.x, r2.y, r3.x, r3.y};
    return out;
}

// One chunk = 16 weight rows x 128 k, as a wave holds it.
template <bool Q4>
struct ChunkRegs {
    uint4 q0, q1;  // q1 only for Q8_0
    uint2 s;       // the lane's row: 4 block scales (f16)
};

template <bool Q4>
__device__ __forceinline__ void load_chunk(ChunkRegs<Q4> &r, const uint4 *__restrict__ qs,
                                           const uint2 *__restrict__ ds, uint64_t chunk,
                                           uint32_t lane) {
    if (Q4) {
        r.q0 = load_stream(qs + chunk * 64 + lane);
    } else {
        r.q0 = load_stream(qs + (chunk * 2) * 64 + lane);
        r.q1 = load_stream(qs + (chunk * 2 + 1) * 64 + lane);
    }
    // (the scales are read once per step like the quants: 1.753 -> 1.722 ms per 7B batch-1 step with
    // this load non-temporal too)
    typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
    const u32x2_t sv = __builtin_nontemporal_load((const u32x2_t *)(ds + chunk * 16 + (lane & 15)));
    r.s = make_uint2(sv.x, sv.y);
}

// How the activation block reaches the matrix cores in gemv_quad_kernel.
enum { X_LDS = 1,     // xq: each wave copies its own pieces into LDS
       X_LAYERNORM = 2, X_RMSNORM = 3,    // f32 residual rows normalised while staged into LDS
       X_RMSPRE = 4 };  // rows that their producer stored as h * scale: times 1 / rms while staged

struct XArgs {
    const uint4 *xq;      // X_LDS
    const float *h;       // X_*NORM: [batch, k]; X_RMSPRE: the rows times the norm's scale
    const float *nscale, *nbias;
    const float2 *stats;  // X_*NORM: [batch][ceil(k/16)] {sum, M2} records of h
    float eps;
    uint32_t k;           // logical reduction length
};

// The same normalisation as a launch of its own, for all batches of 5 to 16 (and of 3 and 4 on wide rows, and of up to 4
// whose rows do not fit gemv_quad_kernel's LDS): row b of h -> xq, statistics merged from the producer's records
// (no reduction over the row).  Grid (k pieces / 256, batch); every wave merges its row's records.
// Bound by one trip to memory behind the launch: everything is requested at once, and the wave's sums are register moves.
template <bool RMS>
__global__ __launch_bounds__(256) void norm_from_stats_kernel(const float *__restrict__ h,
                                                              const float2 *__restrict__ stats,
                                                              const float *__restrict__ nscale,
                                                              const float *__restrict__ nbias,
                                                              float eps, uint32_t k, uint32_t k_pad,
                                                              uint32_t bp, uint4 *__restrict__ xq) {
    constexpr int SREC = 4;  // records a lane holds (k <= 4096); the others are read again
    const uint32_t lane = threadIdx.x & 63, b = blockIdx.y, nt = (k + 15) / 16;
    const uint32_t kp = blockIdx.x * 256 + threadIdx.x;  // piece = 8 consecutive k
    const uint32_t kk = kp * 8, kc = kk < k ? kk : 0;    // k % 8 == 0
    const float2 *row = stats + (uint64_t)b * nt;
    float2 rec[SREC];
#pragma unroll
    for (int u = 0; u < SREC; u++) rec[u] = row[min(lane + 64 * u, nt - 1)];
    const float4 a0 = *(const float4 *)(h + (uint64_t)b * k + kc), a1 = *(const float4 *)(h + (uint64_t)b * k + kc + 4);
    const float4 s0 = *(const float4 *)(nscale + kc), s1 = *(const float4 *)(nscale + kc + 4);
    const float *nb = RMS ? nscale : nbias;
    const float4 b0 = *(const float4 *)(nb + kc), b1 = *(const float4 *)(nb + kc + 4);
    __builtin_amdgcn_sched_barrier(0);
    auto row_sum = [](float t) { return xor32_sum(xor16_sum(group_sum<16>(t))); };
    const float rk = __builtin_amdgcn_rcpf((float)k);
    float mean = 0.f;
    if (!RMS) {
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < SREC; u++) s += lane + 64 * u < nt ? rec[u].x : 0.f;
        for (uint32_t t = lane + 64 * SREC; t < nt; t += 64) s += row[t].x;
        mean = row_sum(s) * rk;
    }
    const uint32_t tail = k & 15;
    const float rc_tail = tail ? __builtin_amdgcn_rcpf((float)tail) : 0.0625f;
    float q = 0.f;
    auto spread = [&](const float2 &r, uint32_t t) {
        const bool last = tail && t == nt - 1;
        const float d = r.x * (last ? rc_tail : 0.0625f) - mean;
        return fmaf((last ? (float)tail : 16.f) * d, d, r.y);
    };
#pragma unroll
    for (int u = 0; u < SREC; u++) q += lane + 64 * u < nt ? spread(rec[u], lane + 64 * u) : 0.f;
    for (uint32_t t = lane + 64 * SREC; t < nt; t += 64) q += spread(row[t], t);
    const float rsd = __builtin_amdgcn_rsqf(row_sum(q) * rk + eps);
    if (kp >= k_pad / 8) return;
    uint4 o = make_uint4(0, 0, 0, 0);
    if (kk < k) {
        const float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        const float sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
        const float bi[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
        float y[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            y[u] = (v[u] - mean) * (sc[u] * rsd);
            if (!RMS) y[u] += bi[u];
        }
        union { uint4 u; half2_t h2[4]; } cv;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            cv.h2[u].x = (_Float16)y[2 * u];
            cv.h2[u].y = (_Float16)y[2 * u + 1];
        }
        o = cv.u;
    }
    xq[(uint64_t)kp * bp + b] = o;
}

int launch_norm_from_stats(const NormFuse &nf, uint64_t batch, uint64_t k, uint64_t k_pad, __half *xq,
                           hipStream_t st) {
    if (!nf.stats || (k & 7))
        return fail(COEUS_INVALID_INPUT, "norm from statistics needs the records and k %% 8 == 0");
    const uint32_t bp = pad_batch(batch);
    const dim3 grid((unsigned)ceil_div(k_pad / 8, 256), (unsigned)batch);
    if (nf.kind == COEUS_NORM_RMSNORM)
        hipLaunchKernelGGL(norm_from_stats_kernel<true>, grid, dim3(256), 0, st, nf.h, nf.stats, nf.scale, nf.bias, nf.eps, (uint32_t)k, (uint32_t)k_pad, bp, (uint4 *)xq);
    else
        hipLaunchKernelGGL(norm_from_stats_kernel<false>, grid, dim3(256), 0, st, nf.h, nf.stats, nf.scale, nf.bias, nf.eps, (uint32_t)k, (uint32_t)k_pad, bp, (uint4 *)xq);
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// ---------------------------------------------------------------- batches of 3 to 16
// Bound by the trips to memory that a wave makes one behind the other and, for long reductions, by the activation rows
// that every workgroup reads from L2 (16 rows x 11008 x 2 B = 352 KB next to 99 KB of Q4_0 weights).  So nothing is staged:
// a wave asks for the four activation fragments of its chunk and for the chunk's weights in its TPW tiles at once, 16 bytes
// a lane each, and multiplies as they arrive; a fragment is read once per workgroup and serves TPW products.  Matrix-core
// roles: A = activations (row = batch entry), B = weights (column = weight row), so lane (j = lane % 16, ig = lane / 16)
// ends up with the results of weight row j for batch entries 4 ig .. 4 ig + 3, and a block's scale is ONE value per lane.
// The waves' sums meet in LDS, every fourth added up and then the four: added one behind the other twelve waves were further off
// than fewer waves with longer shares (2048 x 8192, 16 rows, Q4_0, root mean square error 8.6e-8 of the result's, 7.2e-8 so).  Every
// thread then finishes outputs of its own, whose residual and bias were requested at the start.  Chains of real shapes, one job,
// us a launch with the launch in front (before: activations
// staged in LDS where they fit in 48 KiB, two to six chunks a wave in flight, sums and epilogue on one wave a tile):
//   16 rows, Q4_0: 4096 x 12288 14.2 -> 11.8, 4096 x 4096 9.2 -> 8.6, 4096 x 22016 gated 20.9 -> 16.3, 11008 x 4096 15.6 -> 14.3
//    8 rows, Q8_0: 768 x 2304 6.8 -> 6.0, 768 x 768 7.6 -> 6.0, 768 x 3072 7.2 -> 6.5, 3072 x 768 9.1 -> 7.2, 768 x 50257 14.4 -> 12.6
// 3 and 4 rows (before: gemv_quad_kernel, whose offset term costs every row as much as the products do, and whose sums cancel it: error
// against 64 bits 2.3e-6 of the result for Q4_0 and 2-7e-7 for Q8_0, 6e-8 - 1.1e-7 so), 4 rows, Q4_0: 4096 x 22016 20.6 -> 15.2, 11008 x 4096
// 15.1 -> 12.5, 8192 x 2048 10.3 -> 9.5, 2048 x 8192 7.8 -> 6.9, 2048 x 32000 15.2 -> 12.7; Q8_0: 11008 x 4096 16.3 -> 14.1, 4096 x 12288 15.1
// -> 13.8.  Two chunks of a wave in flight instead of one changed nothing (11008 x 4096 12.2 and 13.0, 8192 x 2048 9.2 and 9.5 us).
// W16 (prompts): a weight is its f16(q d), as in every other prompt matmul, one rounding of the exact product; a chunk's blocks add
// up in the matrix cores, and a wave's chunks behind them (error to 64 bits of 11008 x 4096 Q4_0, 16 rows: 2.0e-7 all in one chain, 1.07e-7 so, 1.69e-7 of the kernel for 17 to 64).
template <bool Q4, int BP, int TPW, bool W16>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4, 8)))
void gemv_rows_kernel(const uint4 *__restrict__ qs, const uint2 *__restrict__ ds, const uint4 *__restrict__ xq, uint32_t ngroups,
                      uint32_t tiles, uint32_t batch, EpiArgs e) {
    // 16-byte pieces from one eight of k to the next, and from row to row: of the interchange format, or of rows gemm_ld(k) elements apart
    const uint32_t xk = W16 ? 1 : BP, xr = W16 ? ngroups * 16 + 8 : 1;
    static_assert(BP == 4 || BP == 8 || BP == 16, "batch padded to 4, 8 or 16");
    static_assert(gemm_ld(128) == 192, "rows of a prompt");
    extern __shared__ float rows_red[];  // [TPW][nwaves][4][64]
    const uint32_t lane = threadIdx.x & 63, nwaves = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t T0 = blockIdx.x * TPW, j = lane & 15, ig = lane >> 4, xb = W16 ? min(j & (BP - 1), batch - 1) * xr : j & (BP - 1);
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    // Output o of the workgroup = (tile, batch row, column); a thread finishes o = threadIdx.x and every blockDim.x-th behind it.
    constexpr uint32_t OUTS = TPW * 16 * BP;
    const bool gated = e.act == COEUS_EPI_SILU_GATE;
    const uint32_t kvpos = (e.kv_k && !e.kv_rows_per_seq) ? *e.kv_pos : 0u;
    float res_pre, bias_pre;  // of the first output (loads unconditional, from a valid address)
    {
        const uint32_t o = threadIdx.x < OUTS ? threadIdx.x : 0, b = o / 16 % BP;
        const uint64_t col = (uint64_t)(T0 + o / (16 * BP)) * 16 + (o & 15);
        const bool ok = e.residual && !gated && b < batch && col < e.n;
        const float *rp = ok ? e.residual : (const float *)ds, *bp = e.bias ? e.bias : (const float *)ds;
        res_pre = rp[ok ? (uint64_t)b * e.n_eff + col : 0];
        bias_pre = bp[(e.bias && col < e.n) ? col : 0];
    }
    float acc[TPW][4];
    uint64_t cb[TPW];
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        cb[t] = (uint64_t)min(T0 + t, tiles - 1) * ngroups;
#pragma unroll
        for (int i = 0; i < 4; i++) acc[t][i] = 0.f;
    }
#pragma unroll 1
    for (uint32_t G = wave; G < ngroups; G += nwaves) {
        uint4 xv[4];
        ChunkRegs<Q4> r[TPW];
        float4_t chunk[W16 ? TPW : 1];
#pragma unroll
        for (int jj = 0; jj < 4; jj++) xv[jj] = xq[((G * 4 + jj) * 4 + ig) * xk + xb];
#pragma unroll
        for (int t = 0; t < TPW; t++) load_chunk<Q4>(r[t], qs, ds, cb[t] + G, lane);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            if (TPW == 4) __builtin_amdgcn_sched_barrier(0);  // (Q8_0: without it the unpacked operands of two blocks live at once and spill)
            union { uint4 u4; half8_t h; } x;
            x.u4 = xv[jj];
#pragma unroll
            for (int t = 0; t < TPW; t++) {
                const ChunkRegs<Q4> &c = r[t];
                const uint32_t qw[8] = {c.q0.x, c.q0.y, c.q0.z, c.q0.w, Q4 ? 0u : c.q1.x, Q4 ? 0u : c.q1.y,
                                        Q4 ? 0u : c.q1.z, Q4 ? 0u : c.q1.w};
                union { uint2 u2; _Float16 h[4]; } s;
                s.u2 = c.s;
                const half8_t wv = Q4 ? unpack_q4(qw[jj]) : unpack_q8(qw[2 * jj], qw[2 * jj + 1]);
                if constexpr (W16) {
                    chunk[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h, wv * s.h[jj], jj ? chunk[t] : zero, 0, 0, 0);
                    if (jj == 3)
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[t][i] += chunk[t][i];
                    continue;
                }
                const float4_t part = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h, wv, zero, 0, 0, 0);
                const float d = (float)s.h[jj];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t][i] = fmaf(d, part[i], acc[t][i]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < TPW; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) rows_red[((t * nwaves + wave) * 4 + i) * 64 + lane] = acc[t][i];
    lds_barrier();
    // q|k|v of sizes that are no multiples of 16: a tile may hold columns of two parts or heads
    const bool kv_odd = e.kv_k && ((e.kv_inner | e.kv_hd) & 15u);
    for (uint32_t o = threadIdx.x; o < OUTS; o += nwaves * 64) {  // (whole waves: OUTS is a multiple of 64)
        const uint32_t t = o / (16 * BP), b = o / 16 % BP, T = T0 + t;
        const uint64_t col = (uint64_t)T * 16 + (o & 15);
        const float *mine = rows_red + (t * nwaves * 4 + (b & 3)) * 64 + (b >> 2) * 16 + (o & 15);
        float part[4] = {0.f, 0.f, 0.f, 0.f};
        uint32_t w = 0;
        for (; w + 4 <= nwaves; w += 4, mine += 1024)
#pragma unroll
            for (uint32_t u = 0; u < 4; u++) part[u] += mine[u * 256];
        if (w < nwaves) part[0] += mine[0];
        if (w + 1 < nwaves) part[1] += mine[256];
        if (w + 2 < nwaves) part[2] += mine[512];
        float v = (part[0] + part[1]) + (part[2] + part[3]);
        const bool live = b < batch && col < e.n, first = o == threadIdx.x;
        if (e.kv_k && (kv_odd || T * 16 >= e.kv_inner)) {
            if (live) epi_store<true>(e, b, col, v, first, res_pre, !e.kv_rows_per_seq, kvpos);
            continue;
        }
        if (e.bias) v += first ? bias_pre : live ? e.bias[col] : 0.f;
        if (gated) {
            // weight rows (2m, 2m+1) = (gate_m, up_m) sit in neighbouring lanes
            const float up = lane_xor1(v);
            if (live && (o & 1) == 0) {
                const uint64_t m = col >> 1;
                float g = silu_f32(v) * up;
                if (e.residual) g += e.residual[(uint64_t)b * e.n_eff + m];
                if (e.out_f32) e.out_f32[(uint64_t)b * e.n_eff + m] = g;
                if (e.out_xq) e.out_xq[xq_index(m, b, e.bp_out)] = __float2half_rn(g);
                if (e.out_lp) e.out_lp[(uint64_t)b * e.lp_ld + m] = f32_to_lp_bits(g, e.lp_bf16);
            }
            continue;
        }
        if (e.act == COEUS_EPI_GELU) v = gelu_f32(v);
        if (e.residual) v += first ? res_pre : live ? e.residual[(uint64_t)b * e.n_eff + col] : 0.f;
        if (live) {
            if (e.out_f32) e.out_f32[(uint64_t)b * e.n_eff + col] = v;
            if (e.out_xq) e.out_xq[xq_index(col, b, e.bp_out)] = __float2half_rn(v);
            if (e.out_lp) e.out_lp[(uint64_t)b * e.lp_ld + col] = f32_to_lp_bits(v, e.lp_bf16);
        }
        if (e.stats_out) {  // uniform; never combined with the gated epilogue
            const uint32_t left = (uint32_t)e.n - T * 16;  // (a tile past the end: unused)
            const float2 r = group16_stats(live ? v : 0.f, live, left < 16 ? left : 16u);
            if ((o & 15) == 0 && live) e.stats_out[(uint64_t)b * e.stats_tiles + T] = r;
        }
    }
}

// ---------------------------------------------------------------- quad kernel (batches of up to 4)
// The decode matmul for batches of 1 and 2, and of 3 and 4 where gemv_takes_rows says no, where a launch is a transient: the whole matrix (10-70 MB) is
// requested within the first microsecond and the kernel ends when the last line has arrived, so
// what counts is that every wave asks for its weights at once, that as few other bytes as possible
// go through the CU's memory pipeline, and that little is left to do after the last line.  A wave
// owns "quads" of four consecutive 128-k chunks of its workgroup's tile (4 KiB of Q4_0 quants per
// quad) and does everything for them on its own:
//   * it requests, in this order, the activations of exactly its quads (or, with a folded norm,
//     the residual values, scale and bias of those k; the row's statistics records are read by
//     wave 0 alone), the block scales (ONE 8-byte load per lane for a whole quad: lane 16 u + r takes
//     the four scales of row r in chunk u), then the quants; all unconditional, from clamped
//     addresses;
//   * as soon as the activation loads have arrived (the weights are still in flight) it
//     normalises / copies them into its PRIVATE slice of LDS as f16 matrix-core fragments; no
//     workgroup barrier orders this (the one barrier of a folded norm hands out the row statistics):
//     a wave only ever reads fragments that it wrote itself;
//   * the quants enter the matrix cores as they are stored: a masked nibble (or a byte) IS the bit
//     pattern of the f16 subnormal n * 2^-24, which v_mfma_f32_16x16x32_f16 multiplies exactly, so
//     a 32-k block costs one shift and four ANDs instead of the conversion to q - 8.  Nibbles kept
//     at bit 4 count 16-fold; the activations of those k positions are staged divided by 16.  The
//     offset comes back through the block's activation sum S: d * (sum x n - 8 S) = sum x (n - 8) d;
//   * chunk u of a quad is multiplied by all 64 lanes (activations replicated over the 16 A rows by
//     row % BP), but only the lanes 16 u .. 16 u + 15 add the scaled block result to their
//     accumulators, because they are the ones that hold chunk u's scales; the four lane groups are
//     summed once at the end.
// The waves' partial sums meet in LDS (16 floats per wave and batch row), and wave 0 adds them up
// and runs the epilogue with one output element per lane (lane = 16 b + column), on operands
// (residual element, cache position) that were requested at kernel start.
template <bool Q4>
__device__ __forceinline__ half8_t quad_operand(uint32_t w0, uint32_t w1) {
    union { uint32_t u[4]; half8_t h; } o;
    if (Q4) {  // nibble positions [k0,k2,k4,k6,k1,k3,k5,k7]: (k0,k1) (k2,k3)<<4 (k4,k5) (k6,k7)<<4
        const uint32_t w8 = w0 >> 8;
        o.u[0] = w0 & 0x000F000Fu; o.u[1] = w0 & 0x00F000F0u; o.u[2] = w8 & 0x000F000Fu; o.u[3] = w8 & 0x00F000F0u;
    } else {   // int8 -> q + 128 in the low byte of each half
        const uint32_t l = w0 ^ 0x80808080u, h = w1 ^ 0x80808080u;
        o.u[0] = __builtin_amdgcn_perm(0u, l, 0x0c010c00u); o.u[1] = __builtin_amdgcn_perm(0u, l, 0x0c030c02u);
        o.u[2] = __builtin_amdgcn_perm(0u, h, 0x0c010c00u); o.u[3] = __builtin_amdgcn_perm(0u, h, 0x0c030c02u);
    }
    return o.h;
}

// One staged piece: 8 consecutive k of one batch row as f16.  Returns what goes into LDS (Q4_0: the
// values that meet a nibble kept at bit 4 divided by 16, rounded to f16 once more, which only changes
// values below 2^-10, by at most 2^-21) and adds the piece's share of the block's activation sum.
template <bool Q4>
__device__ __forceinline__ uint4 quad_piece(uint4 piece, float &sum) {
    union { uint4 u; half2_t h2[4]; } o;
    o.u = piece;
    if (Q4) {
        const half2_t r16 = {(_Float16)0.0625f, (_Float16)0.0625f};
        o.h2[1] = o.h2[1] * r16;
        o.h2[3] = o.h2[3] * r16;
        sum = ((float)o.h2[0].x + (float)o.h2[0].y) + ((float)o.h2[2].x + (float)o.h2[2].y) +
              16.f * (((float)o.h2[1].x + (float)o.h2[1].y) + ((float)o.h2[3].x + (float)o.h2[3].y));
    } else {
        sum = ((float)o.h2[0].x + (float)o.h2[0].y) + ((float)o.h2[1].x + (float)o.h2[1].y) +
              ((float)o.h2[2].x + (float)o.h2[2].y) + ((float)o.h2[3].x + (float)o.h2[3].y);
    }
    return o.u;
}

template <bool Q4, int BP, int XMODE, int QPW, int SREC>
__global__ __launch_bounds__((BP == 4 && XMODE != X_LDS) ? 512 : 1024)  // (four rows with a folded norm: k <= 4096, 8 waves)
__attribute__((amdgpu_waves_per_eu((Q4 && BP * QPW == 1 && XMODE != X_LAYERNORM) ? 6 :
                                   (BP * QPW <= 2 || XMODE == X_LDS) ? 4 : 2, 8)))
void gemv_quad_kernel(const uint4 *__restrict__ qs, const uint2 *__restrict__ ds, XArgs xa, uint32_t ngroups,
                      uint32_t tiles, uint32_t batch, EpiArgs e) {
    static_assert(BP == 1 || BP == 2 || BP == 4, "batch padded to 1, 2 or 4");
    // NORM: f32 rows are normalised while staged; PRE: rows already multiplied by the scale (RMSNorm)
    constexpr bool PRE = XMODE == X_RMSPRE, NORM = XMODE == X_LAYERNORM || XMODE == X_RMSNORM || PRE;
    constexpr bool RMS = XMODE == X_RMSNORM || PRE;
    static_assert(!NORM || QPW == 1, "a folded norm stages one quad per wave");
    constexpr int NI = BP;
    constexpr int WSTRIDE = QPW * BP * 68;  // uint4 per wave: 64 pieces and 16 block sums per quad and batch row
    extern __shared__ uint4 smem[];         // [nwaves][WSTRIDE], partial sums [nwaves][NI][16], row statistics [BP]
    const uint32_t lane = threadIdx.x & 63, nwaves = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15, ig = lane >> 4;
    const uint32_t T = blockIdx.x, nquads = (ngroups + 3) / 4;
    uint4 *xw = smem + wave * WSTRIDE;
    float *sw = (float *)(xw + QPW * BP * 64);  // [QPW][16 blocks][BP]: -8 (or -128) * the block's activation sum
    float *red = (float *)(smem + nwaves * WSTRIDE);
    float2 *rowstat = (float2 *)(red + nwaves * NI * 16);  // {mean, 1 / standard deviation} per batch row

    const uint32_t k = xa.k, nt = (k + 15) / 16;
    // a folded norm: wave 0 also merges the producer's statistics records of the rows (requested first)
    float2 rec0[NORM ? BP : 1][NORM ? SREC : 1];
    if constexpr (NORM) {
        if (wave == 0) {
#pragma unroll
            for (int b = 0; b < BP; b++) {
                const uint32_t bc = (uint32_t)b < batch ? b : 0;
#pragma unroll
                for (int u = 0; u < SREC; u++) rec0[b][u] = xa.stats[(uint64_t)bc * nt + min(lane + 64 * u, nt - 1)];
            }
        }
    }

    // 0. What the epilogue needs is requested now, so that nothing at the end of the kernel waits for
    // a load of its own: the operands of lane (b = ig, column j), by every wave though only wave 0
    // uses them (a load under a branch would make the compiler wait for every request at once).
    float *out_f32 = e.out_f32;
    __half *out_xq = e.out_xq;
    uint16_t *out_lp = e.out_lp;
    float2 *stats_out = e.stats_out;
    void *kv_k = e.kv_k, *kv_v = e.kv_v;
    uint32_t ep_act = e.act, bp_out = e.bp_out, kv_dtype = e.kv_dtype, kv_inner = e.kv_inner, stats_tiles = e.stats_tiles,
             lp_ld = e.lp_ld, lp_bf16 = e.lp_bf16;
    uint64_t ep_n = e.n, n_eff = e.n_eff;
    const uint64_t col = (uint64_t)T * 16 + j;
    const bool gated = ep_act == COEUS_EPI_SILU_GATE;
    const uint32_t kvpos = e.kv_pos ? *e.kv_pos : 0u;
    float res_pre, bias_pre, gs_pre;
    {
        const float *gp = e.g_out ? e.g_scale : (const float *)ds;
        gs_pre = gp[(e.g_out && col < ep_n) ? col : 0];
        const float *rp = (e.residual && !gated) ? e.residual : (const float *)ds;
        const bool ok = e.residual && !gated && ig < batch && col < ep_n;
        res_pre = rp[ok ? (uint64_t)ig * n_eff + col : 0];
        res_pre = ok ? res_pre : 0.f;
        const float *bp = e.bias ? e.bias : (const float *)ds;
        bias_pre = bp[(e.bias && col < ep_n) ? col : 0];
        bias_pre = e.bias ? bias_pre : 0.f;
    }
    // q|k|v: a tile lies inside one head of one of the three parts when both sizes are multiples
    // of 16; where its 16 outputs go in the cache is worked out here, off the tail
    const bool kv_odd = kv_k && ((kv_inner | e.kv_hd) & 15u);
    const bool kv_tile = kv_k && !kv_odd && T * 16 >= kv_inner;
    uint64_t kv_idx = 0;

    float acc[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) acc[i] = 0.f;
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    const uint64_t cb = (uint64_t)T * ngroups;

    for (uint32_t qb = 0; qb < nquads; qb += nwaves * QPW) {  // (a folded norm: exactly one pass)
        const uint32_t q0 = qb + wave * QPW;
        // ---- 1. activations of this wave's quads: lane (u = ig, piece j) of chunk 4 q + u
        uint4 xr[QPW][BP];
        float4 hv[NORM ? BP : 1][2], scv[2], biv[2];
        if constexpr (NORM) {
            const uint32_t G = 4 * q0 + ig;
            uint32_t kk = (G * 16 + j) * 8;
            kk = (G < ngroups && kk < k) ? kk : 0;  // k % 8 == 0: a piece is all in or all out
#pragma unroll
            for (int b = 0; b < BP; b++) {
                const uint32_t bc = (uint32_t)b < batch ? b : 0;
                hv[b][0] = *(const float4 *)(xa.h + (uint64_t)bc * k + kk);
                hv[b][1] = *(const float4 *)(xa.h + (uint64_t)bc * k + kk + 4);
            }
            if (!PRE) {
                scv[0] = *(const float4 *)(xa.nscale + kk);
                scv[1] = *(const float4 *)(xa.nscale + kk + 4);
            }
            if (!RMS) {
                biv[0] = *(const float4 *)(xa.nbias + kk);
                biv[1] = *(const float4 *)(xa.nbias + kk + 4);
            }
        } else {
#pragma unroll
            for (int s = 0; s < QPW; s++) {
                const uint32_t G = min(4 * (q0 + s) + ig, ngroups - 1);
#pragma unroll
                for (int b = 0; b < BP; b++) xr[s][b] = xa.xq[(G * 16 + j) * BP + b];
            }
        }
        // ---- 2. block scales (one load per quad), then the quants
        uint2 sr[QPW];
        uint4 qa[QPW][4], qb8[Q4 ? 1 : QPW][Q4 ? 1 : 4];
        typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int s = 0; s < QPW; s++) {
            const uint32_t G = min(4 * (q0 + s) + ig, ngroups - 1);
            const u32x2_t sv = __builtin_nontemporal_load((const u32x2_t *)(ds + (cb + G) * 16 + j));
            sr[s] = make_uint2(sv.x, sv.y);
        }
#pragma unroll
        for (int s = 0; s < QPW; s++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint64_t c = cb + min(4 * (q0 + s) + u, ngroups - 1);
                if (Q4) {
                    qa[s][u] = load_stream(qs + c * 64 + lane);
                } else {
                    qa[s][u] = load_stream(qs + (c * 2) * 64 + lane);
                    qb8[Q4 ? 0 : s][Q4 ? 0 : u] = load_stream(qs + (c * 2 + 1) * 64 + lane);
                }
            }
        {   // (no branch here: a branch between the requests and their first use makes the compiler wait for all of them)
            const uint32_t inner = kv_inner ? kv_inner : 16u, hd = e.kv_hd ? e.kv_hd : 16u;
            const uint32_t c = (T * 16) % inner, hh = c / hd, d0 = c % hd;
            kv_idx = (((uint64_t)ig * e.kv_heads + hh) * e.kv_max_ctx + kvpos) * hd + d0 + j;
        }
        // ---- 3. stage this wave's activation pieces (the weights are still on their way)
        if constexpr (NORM) {
            if (wave == 0) {
                // mean = sum(s_t) / k, k * var = sum(M2_t + c_t * (s_t / c_t - mean)^2); with mean = 0 the
                // same expression is sum(x^2), which is what the RMS norm divides by.  Hardware
                // reciprocal and reciprocal square root (1 ulp): the result is rounded to f16.
                const float rk = __builtin_amdgcn_rcpf((float)k);
                const uint32_t tail = k & 15;
                const float rc_tail = tail ? __builtin_amdgcn_rcpf((float)tail) : 0.0625f;
#pragma unroll
                for (int b = 0; b < BP; b++) {
                    float sm = 0.f;
#pragma unroll
                    for (int u = 0; u < SREC; u++) sm += lane + 64 * u < nt ? rec0[b][u].x : 0.f;
                    const float mean = RMS ? 0.f : wave_sum(sm) * rk;
                    float q = 0.f;
#pragma unroll
                    for (int u = 0; u < SREC; u++) {
                        const uint32_t t = lane + 64 * u;
                        const bool last = tail && t == nt - 1;
                        const float c = last ? (float)tail : 16.f, rc = last ? rc_tail : 0.0625f;
                        const float d = rec0[b][u].x * rc - mean;
                        q += t < nt ? fmaf(c * d, d, rec0[b][u].y) : 0.f;
                    }
                    const float rsd = __builtin_amdgcn_rsqf(wave_sum(q) * rk + xa.eps);
                    if (lane == 0) rowstat[b] = make_float2(mean, rsd);
                }
            }
            lds_barrier();
            const uint32_t G = 4 * q0 + ig;
            const bool piece_live = G < ngroups && (G * 16 + j) * 8 < k;
            float sc[8];
            if (PRE) {
#pragma unroll
                for (int u = 0; u < 8; u++) sc[u] = 1.f;
            } else {
                const float t[8] = {scv[0].x, scv[0].y, scv[0].z, scv[0].w, scv[1].x, scv[1].y, scv[1].z, scv[1].w};
#pragma unroll
                for (int u = 0; u < 8; u++) sc[u] = t[u];
            }
#pragma unroll
            for (int b = 0; b < BP; b++) {
                const float2 ms = rowstat[b];
                const float v[8] = {hv[b][0].x, hv[b][0].y, hv[b][0].z, hv[b][0].w,
                                    hv[b][1].x, hv[b][1].y, hv[b][1].z, hv[b][1].w};
                float y[8];
#pragma unroll
                for (int u = 0; u < 8; u++) y[u] = (v[u] - ms.x) * (sc[u] * ms.y);  // scale * (x - mean) / sd (MT:124)
                if (!RMS) {
                    const float bi[8] = {biv[0].x, biv[0].y, biv[0].z, biv[0].w, biv[1].x, biv[1].y, biv[1].z, biv[1].w};
#pragma unroll
                    for (int u = 0; u < 8; u++) y[u] += bi[u];
                }
                union { uint4 u; half2_t h2[4]; } o;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    o.h2[u].x = (_Float16)y[2 * u];
                    o.h2[u].y = (_Float16)y[2 * u + 1];
                }
                if (!(piece_live && (uint32_t)b < batch)) o.u = make_uint4(0, 0, 0, 0);
                float sx;
                xw[(ig * 16 + j) * BP + b] = quad_piece<Q4>(o.u, sx);
                sx += dpp_f32<DPP_QUAD_XOR1>(sx);
                sx += dpp_f32<DPP_QUAD_XOR2>(sx);  // the block = four neighbouring pieces
                if ((j & 3) == 0) sw[(ig * 4 + (j >> 2)) * BP + b] = (Q4 ? -8.f : -128.f) * sx;
            }
        } else {
#pragma unroll
            for (int s = 0; s < QPW; s++)
#pragma unroll
                for (int b = 0; b < BP; b++) {
                    float sx;
                    xw[((s * 4 + ig) * 16 + j) * BP + b] = quad_piece<Q4>(xr[s][b], sx);
                    sx += dpp_f32<DPP_QUAD_XOR1>(sx);
                    sx += dpp_f32<DPP_QUAD_XOR2>(sx);
                    if ((j & 3) == 0) sw[((s * 4 + ig) * 4 + (j >> 2)) * BP + b] = (Q4 ? -8.f : -128.f) * sx;
                }
        }
        // ---- 4. products
#pragma unroll
        for (int s = 0; s < QPW; s++) {
            union { uint2 u2; half2_t h[2]; } scu;
            scu.u2 = sr[s];
            const bool chunk_live = 4 * (q0 + s) + ig < ngroups;  // a chunk past the end was re-read: no weight
            float d[4] = {(float)scu.h[0].x, (float)scu.h[0].y, (float)scu.h[1].x, (float)scu.h[1].y};
#pragma unroll
            for (int jj = 0; jj < 4; jj++) d[jj] = chunk_live ? d[jj] : 0.f;
            // this lane group's own chunk: the offset term d * (-8 S) of its four blocks
#pragma unroll
            for (int jj = 0; jj < 4; jj++)
#pragma unroll
                for (int i = 0; i < NI; i++) acc[i] = fmaf(d[jj], sw[((s * 4 + ig) * 4 + jj) * BP + i], acc[i]);
            float dm[4];  // the nibbles entered as n * 2^-24
#pragma unroll
            for (int jj = 0; jj < 4; jj++) dm[jj] = d[jj] * 16777216.f;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t qw[8] = {qa[s][u].x, qa[s][u].y, qa[s][u].z, qa[s][u].w,
                                        Q4 ? 0u : qb8[Q4 ? 0 : s][Q4 ? 0 : u].x, Q4 ? 0u : qb8[Q4 ? 0 : s][Q4 ? 0 : u].y,
                                        Q4 ? 0u : qb8[Q4 ? 0 : s][Q4 ? 0 : u].z, Q4 ? 0u : qb8[Q4 ? 0 : s][Q4 ? 0 : u].w};
#pragma unroll
                for (int jj = 0; jj < 4; jj++) {
                    union { uint4 u4; half8_t h; } xv;
                    xv.u4 = xw[((s * 4 + u) * 16 + 4 * jj + ig) * BP + (j & (BP - 1))];
                    const half8_t wv = Q4 ? quad_operand<true>(qw[jj], 0u) : quad_operand<false>(qw[2 * jj], qw[2 * jj + 1]);
                    const float4_t part = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv.h, wv, zero, 0, 0, 0);
                    if (ig == (uint32_t)u) {
#pragma unroll
                        for (int i = 0; i < NI; i++) acc[i] = fmaf(dm[jj], part[i], acc[i]);
                    }
                }
            }
        }
    }

    // ---- 5. the four lane groups, then the waves, meet; wave 0 finishes the tile
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const float v = xor32_sum(xor16_sum(acc[i]));
        if (ig == 0) red[(wave * NI + i) * 16 + j] = v;
    }
    lds_barrier();
    if (wave != 0) return;
    const uint32_t b = ig;  // this lane's batch row
    float a = 0.f;
    if (b < (uint32_t)NI)
        for (uint32_t w = 0; w < nwaves; w++) a += red[(w * NI + b) * 16 + j];
    const bool live = b < (uint32_t)NI && b < batch && col < ep_n;
    if (kv_odd) {  // q|k|v of sizes that are not multiples of 16: the general walk
        if (live) epi_store<true>(e, b, col, a, true, res_pre, true, kvpos);
        return;
    }
    a += bias_pre;
    if (gated) {
        // weight rows (2m, 2m+1) = (gate_m, up_m) sit in neighbouring lanes
        const float up = lane_xor1(a);
        if (live && (lane & 1) == 0) {
            const uint64_t m = col >> 1;
            float v = fast_silu(a) * up;
            if (e.residual) v += e.residual[(uint64_t)b * n_eff + m];
            if (out_f32) out_f32[(uint64_t)b * n_eff + m] = v;
            if (out_xq) out_xq[xq_index(m, b, bp_out)] = __float2half_rn(v);
            if (out_lp) out_lp[(uint64_t)b * lp_ld + m] = f32_to_lp_bits(v, lp_bf16);
        }
        return;
    }
    if (kv_tile) {  // key or value columns: into the cache, nothing else
        if (live) kv_cache_store(T * 16 < 2 * kv_inner ? kv_k : kv_v, kv_dtype, kv_idx, a);
        return;
    }
    if (ep_act == COEUS_EPI_GELU) a = fast_gelu(a);
    const float v = a + res_pre;
    const uint64_t oidx_g = (uint64_t)b * n_eff + col;
    if (live) {
        if (out_f32) out_f32[(uint64_t)b * n_eff + col] = v;
        if (out_xq) out_xq[xq_index(col, b, bp_out)] = __float2half_rn(v);
        if (out_lp) out_lp[(uint64_t)b * lp_ld + col] = f32_to_lp_bits(v, lp_bf16);
        if (e.g_out) e.g_out[oidx_g] = v * gs_pre;  // the copy that the next norm's matmul stages
    }
    if (stats_out) {  // uniform; never combined with the gated epilogue
        const uint32_t left = (uint32_t)ep_n - T * 16;
        const float2 r = group16_stats(live ? v : 0.f, live, left < 16 ? left : 16u);
        if (j == 0 && b < (uint32_t)NI && b < batch) stats_out[(uint64_t)b * stats_tiles + T] = r;
    }
}

static const size_t kXLdsLimit = 48 * 1024;

bool gemv_can_fuse_norm(const Weight &w, uint64_t batch) {
    if (w.dtype < COEUS_W_Q8_0 || batch < 1 || batch > 16) return false;
    const uint32_t bp = pad_batch(batch);
    // (gemv_quad_kernel: one quad of 512 k per wave, at most 16 waves; 4 or 8 statistics records
    // per lane and row, 8 only for up to two rows)
    return bp <= 4 && (w.k & 7) == 0 && w.k <= 16u * 64u * 8u && w.k_pad * bp * 2 <= kXLdsLimit &&
           (bp < 4 || w.k <= 16u * 64u * 4u);
}

// Batches of 3 and 4, the norm as a launch of its own in front of gemv_rows_kernel instead of folded into gemv_quad_kernel, whose
// four rows every workgroup normalises again.  Decode steps of 4 sequences, ms for 24 - 32 of them, folded / apart: 1B (2048 wide, 24 layers)
// Q4_0 45.6 / 43.6 with the prompt, 7B (4096) 48.75 / 44.2 with the prompt; 12 layers of 1536 Q4_0 15.3 / 14.4, Q8_0 15.2 / 14.8, of 1024
// Q4_0 13.3 / 13.2, Q8_0 13.3 / 13.2 (no difference), of 768 Q8_0 11.5 / 12.1.
bool gemv_norm_apart(const Weight &w, uint64_t batch) { return w.dtype >= COEUS_W_Q8_0 && batch > 2 && w.k >= 1536; }

struct GemvLaunch {
    dim3 grid, block;
    size_t lds;
    hipStream_t st;
    const uint4 *qs;
    const uint2 *ds;
    XArgs xa;
    uint32_t ngroups, tiles, batch;
    EpiArgs e;
};

template <bool Q4, int BPV, int MODE, int QPWV, int SRECV>
static bool quad_launch_one(const GemvLaunch &L) {
    const void *kern = (const void *)gemv_quad_kernel<Q4, BPV, MODE, QPWV, SRECV>;
    if (L.lds > 48 * 1024) {
        static const hipError_t once = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (once != hipSuccess) return false;
    }
    hipLaunchKernelGGL((gemv_quad_kernel<Q4, BPV, MODE, QPWV, SRECV>), L.grid, L.block, L.lds, L.st, L.qs, L.ds, L.xa,
                       L.ngroups, L.tiles, L.batch, L.e);
    return true;
}

template <bool Q4, int BPV>
static bool quad_launch_bp(int xmode, uint32_t qpw, uint32_t srec, const GemvLaunch &L) {
    if (xmode == X_LDS) return qpw == 1 ? quad_launch_one<Q4, BPV, X_LDS, 1, 4>(L) : quad_launch_one<Q4, BPV, X_LDS, 2, 4>(L);
    if (qpw != 1) return false;
    if (xmode == X_LAYERNORM) {
        if (srec == 4) return quad_launch_one<Q4, BPV, X_LAYERNORM, 1, 4>(L);
        if constexpr (BPV <= 2) return quad_launch_one<Q4, BPV, X_LAYERNORM, 1, 8>(L);
        return false;
    }
    if (xmode == X_RMSPRE) {
        if (srec == 4) return quad_launch_one<Q4, BPV, X_RMSPRE, 1, 4>(L);
        if constexpr (BPV <= 2) return quad_launch_one<Q4, BPV, X_RMSPRE, 1, 8>(L);
        return false;
    }
    if (srec == 4) return quad_launch_one<Q4, BPV, X_RMSNORM, 1, 4>(L);
    if constexpr (BPV <= 2) return quad_launch_one<Q4, BPV, X_RMSNORM, 1, 8>(L);
    return false;
}

// Batches of up to 4 that gemv_takes_rows leaves: gemv_quad_kernel, one workgroup per tile of 16 rows.  A wave takes quads of
// four chunks; with a folded norm one quad per wave and as many waves as the reduction has quads;
// plain activations: one or two quads in flight per wave, several passes when 16 waves do not cover
// k that way.
template <bool Q4>
static int launch_gemv_quad(const Weight &w, const __half *xq, uint64_t batch, const EpiArgs &e, hipStream_t st,
                            const NormFuse *nf) {
    const uint32_t ngroups = (uint32_t)(w.k_pad / 128), tiles = (uint32_t)(w.n_pad / 16);
    const uint32_t bp = pad_batch(batch), nquads = (ngroups + 3) / 4;
    if (nf && (!gemv_can_fuse_norm(w, batch) || !nf->stats))
        return fail(COEUS_INVALID_INPUT, "norm fusion needs the activations to fit in LDS and the "
                                         "producer's statistics records");
    if (e.stats_out && e.act == COEUS_EPI_SILU_GATE)
        return fail(COEUS_INVALID_INPUT, "statistics records are not produced by the gated epilogue");
    XArgs xa{};
    xa.xq = (const uint4 *)xq;
    xa.k = (uint32_t)w.k;
    int xmode = X_LDS;
    uint32_t qpw = 1, waves = nquads, srec = 4;
    if (nf) {
        xmode = nf->kind == COEUS_NORM_RMSNORM ? X_RMSNORM : X_LAYERNORM;
        xa.h = nf->h; xa.nscale = nf->scale; xa.nbias = nf->bias; xa.stats = nf->stats; xa.eps = nf->eps;
        srec = w.k > 16u * 64u * 4u ? 8 : 4;
        if (nf->g) {
            if (xmode != X_RMSNORM) return fail(COEUS_INVALID_INPUT, "pre-scaled rows are for a root-mean-square norm");
            xmode = X_RMSPRE;
            xa.h = nf->g;
        }
    } else if (nquads > 16) {
        qpw = 2;
        const uint32_t passes = (nquads + 31) / 32;
        waves = (nquads + 2 * passes - 1) / (2 * passes);
    }
    // every wave keeps its activation pieces in LDS: at most 64 KiB of them per workgroup
    const size_t wbytes = (size_t)qpw * bp * 68 * 16;
    while (waves > 1 && waves * wbytes > 64 * 1024) waves = (waves + 1) / 2;
    GemvLaunch L;
    L.grid = dim3(tiles);
    L.block = dim3(waves * 64);
    L.lds = waves * wbytes + (size_t)waves * bp * 16 * 4 + bp * 8;
    L.st = st;
    L.qs = (const uint4 *)w.data;
    L.ds = (const uint2 *)w.scales;
    L.xa = xa;
    L.ngroups = ngroups; L.tiles = tiles; L.batch = (uint32_t)batch;
    L.e = e;
    bool ok;
    switch (bp) {
        case 1: ok = quad_launch_bp<Q4, 1>(xmode, qpw, srec, L); break;
        case 2: ok = quad_launch_bp<Q4, 2>(xmode, qpw, srec, L); break;
        default: ok = quad_launch_bp<Q4, 4>(xmode, qpw, srec, L); break;
    }
    if (!ok) return fail(COEUS_INVALID_INPUT, "decode matmul: no quad kernel for mode %d and %u quads per wave", xmode, qpw);
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// Batches of 3 and 4, rows as they are: gemv_rows_kernel or gemv_quad_kernel.  Over 185 sizes (512 - 14336 by 256 - 32000; 3 and 4 rows
// alike) the former took, as a share of the latter's time: Q4_0 0.67 - 0.98 everywhere; Q8_0 0.79 - 0.95 on more than 256 tiles (a workgroup
// takes several), and on up to 256 tiles by the waves that the quads, 512 of k each, are: two and a little over 0.92 - 0.99 (1024 0.92 - 0.95, 1056 - 1152 0.95 - 0.99),
// three and four 0.98 - 1.03 (1280 - 2048), five and six 0.87 - 0.95 (2080 - 3072; 3104 0.95, 3584 0.98 and stay), eight to sixteen in one pass, a launch
// that is a single trip, 0.97 - 1.10 (4096 - 8192), several passes 0.73 - 0.98 (beyond 8192).  Narrow rows (k < 1024) belong to models whose norms
// stay folded, and stay with that kernel.
static bool gemv_takes_rows(const Weight &w, uint64_t batch) {
    if (batch > 4) return true;
    if (batch < 3 || w.k < 1024) return false;
    return w.dtype == COEUS_W_Q4_0 || w.n_pad / 16 > 256 || w.k <= 1152 || (w.k > 2048 && w.k <= 3072) || w.k > 8192;
}

// Batches of 3 to 16: tiles and waves of a workgroup of gemv_rows_kernel.  Every workgroup reads all activation rows, so it
// takes as many tiles as leave about a workgroup per CU, six at most (Q8_0 four: registers), else two workgroups per CU;
// waves as many as share the reduction in few trips.  Measured for 8 and 16 rows over 35 matrices of 768 - 5120 wide models
// with 1 - 6 tiles and 2 - 16 waves; the choice is within 4 % of the best of them (4096 x 22016, 16 rows, Q4_0: six tiles 15.9,
// three 17, two 17.4 us; 1536 x 8192: two 6.9, one 7.3; 768 x 50257: two tiles of three waves 12.2, one of six 17.2).
// Few chunks (k <= 512) are few waves, and the outputs of several tiles are more than these finish at once: one tile, a wave per chunk, as long
// as the activations are next to nothing, else two; six tiles only from nine chunks on.  Q4_0, 16 rows, us with as many tiles as above / so: 64 x
// 16400 12.9 / 6.3, x 100000 10.5 / 9.9, 256 x 16400 10.2 / 6.3, x 33000 9.6 / 8.1, 512 x 16400 8.8 / 6.8, x 50257 10.9 / 10.2, 768 x 16400
// 9.3 / 8.0.  400 sizes with 1 - 6 tiles and 1 - 16 waves: 1.3 % above the best of them on average.  (4 rows, 22 sizes: within 3 % of the
// best too, 4096 x 12288 Q4_0 7 %.)
static void gemv_rows_shape(bool q4, uint32_t ngroups, uint32_t tiles, uint32_t &tpw, uint32_t &waves) {
    if (ngroups <= 4 && tiles > 256) {
        tpw = ngroups == 1 || tiles <= (ngroups == 2 ? 2048 : 1536) ? 1 : 2;
        waves = ngroups;
        return;
    }
    tpw = 0;
    for (uint32_t t : {1u, 2u, 3u, 4u, 6u})
        if (!tpw && (t < 6 || (q4 && ngroups > 8)) && ceil_div(tiles, t) <= 256) tpw = t;
    for (uint32_t t : {2u, 3u, 4u})
        if (!tpw && ceil_div(tiles, t) <= 512) tpw = t;
    const bool many = !tpw;
    if (!tpw) tpw = ngroups <= 8 ? 2 : 4;
    waves = (tpw == 3 || tpw == 4) ? 8 : (tpw == 1 && ngroups <= 16) ? 8 : 12;
    if (many && ngroups <= 8) waves = (ngroups + 1) / 2;
    waves = std::min(waves, ngroups);
}

template <bool Q4, int BP, int TPW, bool W16>
static int launch_gemv_rows(const Weight &w, const void *xq, uint32_t batch, uint32_t waves, const EpiArgs &e, hipStream_t st) {
    const size_t lds = (size_t)TPW * waves * 4 * 64 * 4;
    if (lds > 48 * 1024) {
        static const hipError_t once = hipFuncSetAttribute((const void *)gemv_rows_kernel<Q4, BP, TPW, W16>,
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        COEUS_HIP(once);
    }
    const uint32_t ngroups = (uint32_t)(w.k_pad / 128), tiles = (uint32_t)(w.n_pad / 16);
    hipLaunchKernelGGL((gemv_rows_kernel<Q4, BP, TPW, W16>), dim3((uint32_t)ceil_div(tiles, TPW)), dim3(waves * 64), lds, st, (const uint4 *)w.data,
                       (const uint2 *)w.scales, (const uint4 *)xq, ngroups, tiles, batch, e);
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// x: rows of the interchange format, or (W16) plain f16 rows gemm_ld(k) elements apart.
template <bool Q4, bool W16 = false>
static int launch_gemv_rows_of(const Weight &w, const void *x, uint64_t batch, const EpiArgs &e, hipStream_t st) {
    uint32_t tpw, waves;
    gemv_rows_shape(Q4, (uint32_t)(w.k_pad / 128), (uint32_t)(w.n_pad / 16), tpw, waves);
    auto with = [&](auto bp) -> int {
        constexpr int BP = decltype(bp)::value;
        const uint32_t b = (uint32_t)batch;
        switch (tpw) {
            case 1: return launch_gemv_rows<Q4, BP, 1, W16>(w, x, b, waves, e, st);
            case 2: return launch_gemv_rows<Q4, BP, 2, W16>(w, x, b, waves, e, st);
            case 3: return launch_gemv_rows<Q4, BP, 3, W16>(w, x, b, waves, e, st);
            case 4: return launch_gemv_rows<Q4, BP, 4, W16>(w, x, b, waves, e, st);
            default: if constexpr (Q4) return launch_gemv_rows<Q4, BP, 6, W16>(w, x, b, waves, e, st);
        }
        return fail(COEUS_INVALID_INPUT, "decode matmul: no kernel for %u tiles a workgroup", tpw);
    };
    const uint32_t bp = pad_batch(batch);
    return bp <= 4 ? with(std::integral_constant<int, 4>{}) : bp == 8 ? with(std::integral_constant<int, 8>{}) : with(std::integral_constant<int, 16>{});
}

template <bool Q4>
static int launch_gemv_quant(const Weight &w, const __half *xq, uint64_t batch, const EpiArgs &e,
                             hipStream_t st, const NormFuse *nf) {
    // (a folded norm and a pre-scaled copy of the output are gemv_quad_kernel's)
    if (pad_batch(batch) <= 4 && (nf || e.g_out || !gemv_takes_rows(w, batch))) return launch_gemv_quad<Q4>(w, xq, batch, e, st, nf);
    // gemv_rows_kernel on staged f16 activations (the norm is a launch of its own)
    if (nf) return fail(COEUS_INVALID_INPUT, "norm fusion is for batches of up to 4");
    if (e.stats_out && e.act == COEUS_EPI_SILU_GATE)
        return fail(COEUS_INVALID_INPUT, "statistics records are not produced by the gated epilogue");
    return launch_gemv_rows_of<Q4>(w, xq, batch, e, st);
}

// ---------------------------------------------------------------- dense kernel (f32 / bf16)
// One wave per output row.  NORM = 0: x is the activation block [batch, k] in global memory.
// NORM = 1 (LayerNorm) / 2 (RMSNorm): x is the residual stream; the workgroup (16 waves = 16 rows)
// normalises it once into LDS, evaluated like norm_token_kernel (scale * (x - mean) / sd + bias),
// and its waves read the normalised rows from there: no separate norm launch.  Wave b computes
// the statistics of batch row b on its own (two passes over the row), while every wave already
// has its first weights on the way.
// NORM = 3: the norm of the sublayer before stands behind it.  x is the residual stream h, y the
// sublayer's bare output: the workgroup stages h + y / rms(y) * scale (* ls), and the first one stores
// these rows as the new residual stream.  LDS: y rows (then the sums), [2][k] scales, h rows behind them.
struct PostNorm {
    const float *y, *ls;
    float *h_out;
};
// 1 / standard deviation of a whole-slice norm, rounded once: the f32 value and a Newton step in f64 (a square root and a
// division in f64 would spill the rows that wait in registers).
__device__ __forceinline__ float whole_norm_rs(double var, float eps) {
    const double v = var + (double)eps;
    const float r = 1.0f / sqrtf((float)v);
    const double d = r;
    return r > 0.f && r < INFINITY ? (float)(d * fma(-0.5 * v * d, d, 1.5)) : r;
}
// 1 / n to 2^-46, in the registers that a wave has left (see above)
__device__ __forceinline__ double inv_count(uint32_t n) {
    const double r = 1.0f / (float)n;
    return fma(fma(-(double)n, r, 1.0), r, r);
}
// The staging of NORM 1 - 4: rows of x (see above; 4: LayerNorm over all rows together) -> normalised f32 values, element i of row b handed to put(b, i, v)
// (which may write it to xn + b k + i).  Every wave of the workgroup takes part; the last barrier is the caller's.  LDS
// at xn: [BP][k] rows, [2][k] scale and bias, partial sums, statistics (NORM == 3: then [BP][k] residual rows).
// The sums of NORM 4 are carried in f64, as where that norm is a launch of its own (norm_sequence_kernel).
template <int BP, int NORM, class Put>
__device__ __forceinline__ void stage_normed_rows(float *xn, const float *__restrict__ x, uint64_t k, uint32_t batch,
                                                  const float *__restrict__ nscale, const float *__restrict__ nbias, float eps,
                                                  uint64_t ldx, const PostNorm &post, Put put) {
    typedef typename std::conditional<NORM == 4, double, float>::type Sum;
    const uint32_t ld = (uint32_t)k;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
    // One trip to memory: the rows, the scale and the bias all go to LDS first; the two
    // statistics passes and the normalisation then work from there.
    float *gs = xn + (size_t)BP * ld, *bs = gs + k;  // scale, bias
    Sum *red = (Sum *)(bs + k);                     // [16 waves][BP] partial sums (NORM 4: k is a multiple of 32)
    float *stat = (float *)(red + 16 * BP);         // [0][b] mean, [1][b] standard deviation (NORM 4: its reciprocal)
    float *hs = stat + 32;                          // NORM == 3: [BP][k] residual rows
    Sum ps[BP], mean = 0;                           // (mean: NORM 4, unrounded)
#pragma unroll
    for (int b = 0; b < BP; b++) ps[b] = 0;
    for (uint64_t i = threadIdx.x; i < k; i += blockDim.x) {
        gs[i] = nscale[i];
        if (NORM == 1 || NORM == 4) bs[i] = nbias ? nbias[i] : 0.f;
        if (NORM == 3) bs[i] = post.ls ? post.ls[i] : 1.0f;
#pragma unroll
        for (int b = 0; b < BP; b++)
            if (b < (int)batch) {
                const float v = NORM == 3 ? post.y[(uint64_t)b * k + i] : x[(uint64_t)b * ldx + i];
                xn[(uint32_t)b * ld + i] = v;
                if (NORM == 3) hs[(uint32_t)b * ld + i] = x[(uint64_t)b * ldx + i];
                ps[b] += v;
            }
    }
    // every wave's partial per row -> wave 0 finishes row b = lane; NORM 4: every wave finishes all rows together
    auto finish = [&](Sum (&p)[BP]) -> Sum {
#pragma unroll
        for (int b = 0; b < BP; b++) {
            Sum t;
            if constexpr (NORM == 4) t = wave_sum_f64(p[b]);
            else t = wave_sum(p[b]);
            if (lane == 0) red[wave * BP + b] = t;
        }
        __syncthreads();
        Sum tot = 0;
        if (NORM == 4) {
            for (uint32_t i = lane; i < nwaves * BP; i += 64) tot += red[i];  // (zero for the rows that are not there)
            tot = wave_sum_f64(tot);
            __syncthreads();  // (red is written again)
        } else if (wave == 0 && lane < BP) {
            for (uint32_t w = 0; w < nwaves; w++) tot += red[w * BP + lane];
        }
        return tot;
    };
    if (NORM == 4) {
        mean = finish(ps) * inv_count((uint32_t)k * batch);
    } else if (NORM == 1) {
        const Sum tot = finish(ps);
        if (wave == 0 && lane < BP) stat[lane] = tot / (float)k;
        __syncthreads();
    } else if (threadIdx.x < BP) {
        stat[threadIdx.x] = 0.f;  // a root-mean-square norm subtracts no mean
    }
#pragma unroll
    for (int b = 0; b < BP; b++) ps[b] = 0;
    if (NORM == 2 || NORM == 3) __syncthreads();  // the rows and the zero means are in LDS
    for (uint64_t i = threadIdx.x; i < k; i += blockDim.x)
#pragma unroll
        for (int b = 0; b < BP; b++)
            if (b < (int)batch) {
                const Sum d = xn[(uint32_t)b * ld + i] - (NORM == 4 ? mean : (Sum)stat[b]);
                ps[b] = fma(d, d, ps[b]);
            }
    float whole_mean = 0.f, whole_rs = 0.f;
    if constexpr (NORM == 4) {
        whole_mean = (float)mean;
        whole_rs = whole_norm_rs(finish(ps) * inv_count((uint32_t)k * batch), eps);
    } else {
        const Sum tot = finish(ps);
        if (wave == 0 && lane < BP) stat[16 + lane] = sqrtf(tot / (float)k + eps);
        __syncthreads();
    }
    for (uint64_t i = threadIdx.x; i < k; i += blockDim.x) {
        const float g = gs[i], bi = NORM == 1 || NORM == 4 ? bs[i] : 0.f;
#pragma unroll
        for (int b = 0; b < BP; b++)
            if (b < (int)batch) {
                if (NORM == 3) {
                    const float v = fmaf(xn[(uint32_t)b * ld + i] / stat[16 + b] * g, bs[i], hs[(uint32_t)b * ld + i]);
                    put((uint32_t)b, (uint32_t)i, v);
                    if (blockIdx.x == 0) post.h_out[(uint64_t)b * k + i] = v;
                } else if (NORM == 4) {
                    put((uint32_t)b, (uint32_t)i, g * (xn[(uint32_t)b * ld + i] - whole_mean) * whole_rs + bi);
                } else {
                    put((uint32_t)b, (uint32_t)i, g * (xn[(uint32_t)b * ld + i] - stat[b]) / stat[16 + b] + bi);
                }
            }
    }
}

// One plain activation row, k % 8 == 0: R weight rows a wave, D steps of 512 k of each in flight next to the activations they
// share.  Bound by the weights' stream, and where that is short by the trips to memory a wave makes one behind the other.
// Two rows (gemv_many_kernel) against one with two steps at most (gemv_dense_kernel's general form), which reads twice the weights'
// bytes in activations (f32 next to bf16) and leaves memory idle between its steps, us, distinct weights in turn, there /
// here: bf16 4096 x 22016 33.2 / 29.0, x 32000 46.3 / 40.9, x 12352 19.7 / 18.3, 2048 x 11264 11.2 / 9.0, x 2048 4.3 / 3.5;
// f32 4096 x 22016 74.6 / 65.9.  The matrix cores had rows of these: 5632 x 2048 7.7 / 5.5, 11008 x 4096
// 18.4 / 17.7, 4096 x 4096 7.5 / 7.5, 768 x 50257 13.5 / 13.4, 1024 x 16384 7.5 / 6.9.  Four rows a wave with two or three steps:
// 29.9, 40.0, 20.1, 10.1, 4.3; eight are slower than one.
// One row with D steps (gemv_dense_kernel's D) where up to 1024 rows leave compute units without a workgroup of two, against what they
// had: f32 3072 x 768 5.76 / 4.85, 8192 x 1024 11.9 / 9.0, 768 x 3072 4.43 / 4.11, 4096 x 3072 13.3 / 12.8; bf16 3072 x 768 3.81 / 3.39,
// 11008 x 1024 8.3 / 6.9.  A row over two or four waves that meet in LDS: 5.07, 10.1 and 3.49, 7.1 at best.
template <bool BF16, int D, int R>
__device__ __forceinline__ void one_row(const void *__restrict__ wdata, const float *__restrict__ x, uint32_t k, const EpiArgs &e) {
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int Q = BF16 ? 1 : 2;
    const uint32_t n = (uint32_t)e.n, j0 = (blockIdx.x * 4 + wave) * R, trips = (k + 512 * D - 1) / (512 * D);
    uint4 wv[D][R][Q];
    float4 xv[D][2];
    const char *row[R];
#pragma unroll
    for (int r = 0; r < R; r++) row[r] = (const char *)wdata + (uint64_t)min(j0 + r, n - 1) * k * (BF16 ? 2 : 4);
    auto request = [&](int d, uint32_t step) {  // (a lane behind the end re-reads the last 8 and does not use them)
        const uint32_t i = min(512 * step + 8 * lane, k - 8);
        xv[d][0] = *(const float4 *)(x + i);
        xv[d][1] = *(const float4 *)(x + i + 4);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int q = 0; q < Q; q++) wv[d][r][q] = load_stream((const uint4 *)(row[r] + (uint64_t)i * (BF16 ? 2 : 4)) + q);
    };
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.f;
    auto multiply = [&](int d) {
        const float v[8] = {xv[d][0].x, xv[d][0].y, xv[d][0].z, xv[d][0].w, xv[d][1].x, xv[d][1].y, xv[d][1].z, xv[d][1].w};
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint4 a = wv[d][r][0], c = wv[d][r][Q - 1];
            float t[8];
            if (BF16) {
                const uint32_t q[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int u = 0; u < 4; u++) { t[2 * u] = __uint_as_float(q[u] << 16); t[2 * u + 1] = __uint_as_float(q[u] & 0xffff0000u); }
            } else {
                const uint32_t q[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
                for (int u = 0; u < 8; u++) t[u] = __uint_as_float(q[u]);
            }
#pragma unroll
            for (int u = 0; u < 8; u++) acc[r] = fmaf(t[u], v[u], acc[r]);
        }
    };
#pragma unroll
    for (int d = 0; d < D; d++) request(d, d);
    for (uint32_t i = 0; i + 1 < trips; i++) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            __builtin_amdgcn_sched_barrier(0);
            multiply(d);
            __builtin_amdgcn_sched_barrier(0);
            request(d, (i + 1) * D + d);
        }
    }
#pragma unroll
    for (int d = 0; d < D; d++)
        if (512 * ((trips - 1) * D + d) + 8 * lane < k) multiply(d);
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = wave_sum(acc[r]);
    if constexpr (R == 2) {
        if (epi_gated(e.act)) {
            if (lane == 0 && j0 + 1 < n) epi_store_gated(e, 0, j0 / 2, acc[0], acc[1]);
            return;
        }
    }
    if (lane < R && j0 + lane < n) epi_store<true>(e, 0, j0 + lane, lane ? acc[R - 1] : acc[0]);
}

template <bool BF16, int D>
__global__ __launch_bounds__(256) void gemv_many_kernel(const void *__restrict__ wdata, const float *__restrict__ x, uint32_t k, EpiArgs e) {
    one_row<BF16, D, 2>(wdata, x, k, e);
}

// D > 0: one plain row, k % 8 == 0, 16-byte pointers, no gate: the code above with a weight row a wave
template <bool BF16, int BP, int NORM, int D = 0>
__global__ __launch_bounds__(D ? 256 : 1024) void gemv_dense_kernel(const void *__restrict__ wdata,
                                                          const float *__restrict__ x, uint64_t k,
                                                          uint32_t batch, EpiArgs e,
                                                          const float *__restrict__ nscale,
                                                          const float *__restrict__ nbias, float eps,
                                                          uint64_t ldx, PostNorm post) {
    if constexpr (D > 0) {
        one_row<BF16, D, 1>(wdata, x, (uint32_t)k, e);
        return;
    }
    extern __shared__ float xn[];  // NORM: [BP][k] rows, [2][k] scale and bias, partial sums, statistics
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
    const uint64_t j = (uint64_t)blockIdx.x * nwaves + wave;
    const uint64_t jc = j < e.n ? j : e.n - 1;  // waves past the end repeat the last row (no early
                                                // return: every wave takes part in the barriers)
    float acc[BP];
#pragma unroll
    for (int b = 0; b < BP; b++) acc[b] = 0.f;
    const bool vec = (k & 7) == 0;
    // The first two steps of the row (2 x 512 k) are requested before anything else, from clamped
    // addresses (a step past the end re-reads the last 8 weights and is not used).  Weights are read
    // once per step: non-temporal loads (250M bf16, batch 1: 0.358 -> 0.344 ms per step).
    auto wload = [&](uint64_t k0, uint4 &a, uint4 &b) {
        const uint64_t kc = k0 + 8 <= k ? k0 : k - 8;
        if (BF16) {
            a = load_stream((const uint4 *)((const uint16_t *)wdata + jc * k + kc));
        } else {
            a = load_stream((const uint4 *)((const float *)wdata + jc * k + kc));
            b = load_stream((const uint4 *)((const float *)wdata + jc * k + kc + 4));
        }
    };
    uint4 wa0 = make_uint4(0, 0, 0, 0), wb0 = wa0, wa1 = wa0, wb1 = wa0;
    if (vec) {
        wload((uint64_t)lane * 8, wa0, wb0);
        wload((uint64_t)lane * 8 + 512, wa1, wb1);
    }
    const float *xs = x;  // where the main loop reads activation row b: xs + b * k
    if (NORM) {
        stage_normed_rows<BP, NORM>(xn, x, k, batch, nscale, nbias, eps, ldx, post,
                                    [&](uint32_t b, uint32_t i, float v) { xn[(uint64_t)b * k + i] = v; });
        __syncthreads();
        xs = xn;
    }
    if (vec) {
        auto step = [&](uint64_t k0, const uint4 &ra, const uint4 &rb) {
            float wv[8];
            if (BF16) {
                const uint32_t r[4] = {ra.x, ra.y, ra.z, ra.w};
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    wv[2 * t] = __uint_as_float(r[t] << 16);
                    wv[2 * t + 1] = __uint_as_float(r[t] & 0xffff0000u);
                }
            } else {
                wv[0] = __uint_as_float(ra.x); wv[1] = __uint_as_float(ra.y);
                wv[2] = __uint_as_float(ra.z); wv[3] = __uint_as_float(ra.w);
                wv[4] = __uint_as_float(rb.x); wv[5] = __uint_as_float(rb.y);
                wv[6] = __uint_as_float(rb.z); wv[7] = __uint_as_float(rb.w);
            }
#pragma unroll
            for (int b = 0; b < BP; b++) {
                if (b < (int)batch) {
                    const float4 xa = *(const float4 *)(xs + (uint64_t)b * k + k0);
                    const float4 xb = *(const float4 *)(xs + (uint64_t)b * k + k0 + 4);
                    float s = acc[b];
                    s = fmaf(wv[0], xa.x, s); s = fmaf(wv[1], xa.y, s);
                    s = fmaf(wv[2], xa.z, s); s = fmaf(wv[3], xa.w, s);
                    s = fmaf(wv[4], xb.x, s); s = fmaf(wv[5], xb.y, s);
                    s = fmaf(wv[6], xb.z, s); s = fmaf(wv[7], xb.w, s);
                    acc[b] = s;
                }
            }
        };
        uint64_t k0 = (uint64_t)lane * 8;
        if (k0 < k) step(k0, wa0, wb0);
        if (k0 + 512 < k) step(k0 + 512, wa1, wb1);
        // longer rows: one step ahead
        if (k0 + 1024 < k) {
            k0 += 1024;
            wload(k0, wa0, wb0);
            for (; k0 < k; k0 += 512) {
                wload(k0 + 512, wa1, wb1);
                step(k0, wa0, wb0);
                wa0 = wa1; wb0 = wb1;
            }
        }
    } else {
        for (uint64_t kk = lane; kk < k; kk += 64) {
            const float wv = BF16 ? bf16_bits_to_f32(((const uint16_t *)wdata)[jc * k + kk])
                                  : ((const float *)wdata)[jc * k + kk];
#pragma unroll
            for (int b = 0; b < BP; b++)
                if (b < (int)batch) acc[b] = fmaf(wv, xs[(uint64_t)b * k + kk], acc[b]);
        }
    }
#pragma unroll
    for (int b = 0; b < BP; b++) acc[b] = wave_sum(acc[b]);
    if (epi_gated(e.act)) {
        // pair (gate_m, up_m) = rows (2m, 2m+1) live in neighbouring waves: go through LDS
        __shared__ float pair[16][16];
        if (lane == 0)
#pragma unroll
            for (int b = 0; b < BP; b++) pair[wave][b] = acc[b];
        __syncthreads();
        if ((wave & 1) == 0 && lane < batch && j + 1 < e.n)
            epi_store_gated(e, lane, j / 2, pair[wave][lane], pair[wave + 1][lane]);
        return;
    }
    if (lane == 0 && j < e.n)
#pragma unroll
        for (int b = 0; b < BP; b++)
            if (b < (int)batch) epi_store<true>(e, b, j, acc[b]);
}

// One activation row with the norm in front (NORM 1 or 2), k % 8 == 0, k <= 512 STEPS: no LDS and no barrier.  A wave
// keeps the whole row in registers in the places of its weight loads (lane: 8 consecutive elements of every 512),
// finds the statistics by itself and multiplies R weight rows, all of whose loads are out before the row is
// normalised.  The kernel above normalises once for 16 rows, in five passes through LDS with a barrier behind each:
// 6.9 - 7.1 us for 768 x 2304 and 768 x 3072 in f32 and 6.0 in bf16; here 4.9 - 5.1 and 4.0 - 4.2.
constexpr int kRowR = 4;  // (2: 2-3 % slower steps of the 250M models)
template <bool BF16, bool RMS, int STEPS, int R>
__global__ __launch_bounds__(256) void gemv_row_kernel(const void *__restrict__ wdata, const float *__restrict__ x, uint32_t k,
                                                       const float *__restrict__ nscale, const float *__restrict__ nbias, float eps,
                                                       EpiArgs e) {
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n = (uint32_t)e.n, j0 = (blockIdx.x * 4 + wave) * R;
    float4 xv[STEPS][2], gv[STEPS][2], bv[STEPS][2];
    const float *bp = RMS || !nbias ? nscale : nbias;  // (unused then)
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const uint32_t i = min(512 * s + 8 * lane, k - 8);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            xv[s][h] = *(const float4 *)(x + i + 4 * h);
            gv[s][h] = *(const float4 *)(nscale + i + 4 * h);
            if (!RMS) bv[s][h] = *(const float4 *)(bp + i + 4 * h);
        }
    }
    uint4 wv[R][STEPS][BF16 ? 1 : 2];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t row = min(j0 + r, n - 1);
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            const uint64_t at = (uint64_t)row * k + min(512 * s + 8 * lane, k - 8);
            if (BF16) wv[r][s][0] = load_stream((const uint4 *)((const uint16_t *)wdata + at));
            else {
                wv[r][s][0] = load_stream((const uint4 *)((const float *)wdata + at));
                wv[r][s][BF16 ? 0 : 1] = load_stream((const uint4 *)((const float *)wdata + at + 4));
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    auto row_sum = [](float t) { return xor32_sum(xor16_sum(group_sum<16>(t))); };
    float v[STEPS][8];
    float mean = 0.f, rs;
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const bool in = 512 * s + 8 * lane < k;
        const float t[8] = {xv[s][0].x, xv[s][0].y, xv[s][0].z, xv[s][0].w, xv[s][1].x, xv[s][1].y, xv[s][1].z, xv[s][1].w};
#pragma unroll
        for (int u = 0; u < 8; u++) v[s][u] = in ? t[u] : 0.f;
    }
    if (!RMS) {
        float sum = 0.f;
#pragma unroll
        for (int s = 0; s < STEPS; s++)
#pragma unroll
            for (int u = 0; u < 8; u++) sum += v[s][u];
        mean = row_sum(sum) / (float)k;
    }
    {
        float sq = 0.f;
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            const bool in = 512 * s + 8 * lane < k;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float d = in ? v[s][u] - mean : 0.f;
                sq = fmaf(d, d, sq);
            }
        }
        rs = 1.0f / sqrtf(row_sum(sq) / (float)k + eps);
    }
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const bool in = 512 * s + 8 * lane < k;
        const float g[8] = {gv[s][0].x, gv[s][0].y, gv[s][0].z, gv[s][0].w, gv[s][1].x, gv[s][1].y, gv[s][1].z, gv[s][1].w};
        float b[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (!RMS && nbias) {
            const float t[8] = {bv[s][0].x, bv[s][0].y, bv[s][0].z, bv[s][0].w, bv[s][1].x, bv[s][1].y, bv[s][1].z, bv[s][1].w};
#pragma unroll
            for (int u = 0; u < 8; u++) b[u] = t[u];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) v[s][u] = in ? g[u] * (v[s][u] - mean) * rs + b[u] : 0.f;
    }
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        acc[r] = 0.f;
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            const uint4 a = wv[r][s][0], c = wv[r][s][BF16 ? 0 : 1];
            float w[8];
            if (BF16) {
                const uint32_t q[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int u = 0; u < 4; u++) { w[2 * u] = __uint_as_float(q[u] << 16); w[2 * u + 1] = __uint_as_float(q[u] & 0xffff0000u); }
            } else {
                const uint32_t q[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
                for (int u = 0; u < 8; u++) w[u] = __uint_as_float(q[u]);
            }
            const bool in = 512 * s + 8 * lane < k;  // (a lane behind the end re-read the last weights: an infinite one times 0)
#pragma unroll
            for (int u = 0; u < 8; u++) acc[r] = fmaf(in ? w[u] : 0.f, v[s][u], acc[r]);
        }
        acc[r] = row_sum(acc[r]);
    }
    // lane r finishes row r (gated: lane m the pair 2m, 2m + 1)
    if (epi_gated(e.act)) {
        float g = acc[0], u = acc[R > 1 ? 1 : 0];
#pragma unroll
        for (int m = 1; m < R / 2; m++)
            if (lane == (uint32_t)m) { g = acc[2 * m]; u = acc[2 * m + 1]; }
        if (lane < R / 2 && j0 + 2 * lane + 1 < n) epi_store_gated(e, 0, j0 / 2 + lane, g, u);
    } else {
        float t = acc[0];
#pragma unroll
        for (int r = 1; r < R; r++)
            if (lane == (uint32_t)r) t = acc[r];
        if (lane < R && j0 + lane < n) epi_store<true>(e, 0, j0 + lane, t);
    }
}

// ---------------------------------------------------------------- dense rows on the matrix cores (2 - 16 rows)
// y[b, j] for a tile of 16 weight rows j and all b at once.  bf16 weights: v_mfma_f32_16x16x32_bf16 with the weights as
// they are stored and every activation as the sum of three bf16 (8 mantissa bits each: x exactly), three instructions
// per 32 of k into one f32 accumulator.  f32 weights: v_mfma_f32_16x16x4_f32.  The products are those of the f32 form;
// what changes is the order of the sums.
//
// gemv_dense_kernel (a wave per weight row, activations by f32 FMA) reads `batch` f32 activations per weight: at batch
// 4 that is eight times the weights' bytes, out of L2 where a row does not fit the first-level cache.  Here a tile's
// 16 rows share them, and they are split once per wave.  Us per launch, there / here, distinct weights in turn:
//              batch 2        4            8            16
//   2048 x 2048   5.8 / 4.8    7.4 / 4.9   10.5 / 5.3    16.7 / 6.6
//   5632 x 2048  11.6 / 8.2   15.4 / 8.6   21.9 / 10.7   35.2 / 14.1
//   4096 x 22016   47 / 34     73 / 36      118 / 40      215 / 55
//   768 x 50257    28 / 14     41 / 14       68 / 16      127 / 18
// f32: 768 x 3072 9.0 / 4.4 at batch 8, 768 x 50257 79 / 30, 4096 x 4096 31 / 15.
// (One row: 4.2, 8.7, 33, 18.5 there; where it comes here gemv_uses_mfma says.)  The large ones are
// at 5 TB/s of weights.  A matrix with an infinite value stays there (times a piece that is zero it would be a NaN).
//
// The workgroup's waves take a share of k each, in pairs of 32-wide chunks: a wave request is 8 rows x 128 bytes, as
// the weights lie, and passes through a corner of LDS that is the wave's own to where the matrix cores want it (a
// lane: 8 consecutive k of one row).  Loaded the way they are multiplied (16 rows x 64 bytes, neighbouring lanes in
// different rows) the same weights take a third longer: 4096 x 22016 at batch 4 in 51 against 40 us.  The activations
// travel likewise.  PD pairs are in flight per wave across the ends of tiles; the waves' partial tiles meet in LDS.
//
// Few outputs are few tiles of 16, and a compute unit brings in 50 GB/s alone (f32 3072 x 768: 48 tiles, 257 KB each of weights and
// activations).  Up to eight activation rows leave half of the sixteen columns unused, up to four three quarters, so the lines of a tile can be
// TS parts of k of 16 / TS weight rows and the columns the activations of the same parts: of the product, part i's lines meet part i's
// columns in the blocks on the diagonal, and those are added.  Twice or four times the workgroups for the same instructions.  us, tiles of 16 /
// in parts: f32, 4 rows of 3072 x 768 8.3 / 5.1, 8192 x 1024 16.7 / 9.2, 768 x 768 4.4 / 3.4, 8 of 3072 x 768 8.8 / 6.5; bf16, 4 of 3072 x 768
// 5.7 / 4.7, 8192 x 1024 10.1 / 7.1, 5632 x 2048 10.1 / 8.0, 8 of 2048 x 1024 5.4 / 4.9.

// Two values -> their three bf16, a pair of upper halves per piece.  What is left of an infinity is zero (its own
// difference would be a NaN).
struct Split2 { uint32_t p[3]; };
__device__ __forceinline__ Split2 split2(float a, float b) {
    uint32_t v[2] = {__float_as_uint(a), __float_as_uint(b)};
    Split2 s;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        s.p[i] = __builtin_amdgcn_perm(v[1], v[0], 0x07060302u);
        if (i == 2) break;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float f = __uint_as_float(v[j]), h = __uint_as_float(v[j] & 0xffff0000u);
            v[j] = __float_as_uint(i == 0 && f == h ? 0.f : f - h);
        }
    }
    return s;
}
// The tiles blockIdx.x, + grid, .. of the workgroup.  XQ > 0: f32 activation rows x [batch][k] in global memory, read
// four to a request (XQ requests cover the batch) and split on their way into the wave's corner.  XQ == 0: `stage`,
// which runs behind the first requests, puts them into LDS: piece i of row b at xs.at(i, b).
// k % 64 == 0 and at least one pair of chunks per wave.
// KEEP: a wave's share of k is at most PD pairs, and its split activations stay in registers from tile to tile.
// lds: mfma_wave_lds(XQ) uint4 per wave.
// TS: parts of k (XQ > 0 only, requests for sixteen rows: the columns).  FOLD: sums of bf16 in groups (f32's always are).
// (Rows 16 bytes longer than k: at a multiple of 256 bytes apart they would share their banks.)
struct SplitRows {  // bf16 weights: three pieces
    uint16_t *p;
    uint32_t k, rows;
    static constexpr size_t bytes(size_t rows, size_t k) { return 3 * rows * (k + 8) * 2; }
    __device__ uint16_t *at(int i, uint32_t b) const { return p + (i * rows + b) * (k + 8); }
    __device__ void put(uint32_t b, uint32_t i, float v) const {
        const Split2 s = split2(v, 0.f);
#pragma unroll
        for (int j = 0; j < 3; j++) at(j, b)[i] = (uint16_t)s.p[j];
    }
    __device__ void put4(uint32_t b, uint32_t i, const float4_t &v) const {
        const Split2 lo = split2(v[0], v[1]), hi = split2(v[2], v[3]);
#pragma unroll
        for (int j = 0; j < 3; j++) *(uint2 *)(at(j, b) + i) = make_uint2(lo.p[j], hi.p[j]);
    }
    __device__ void put2(uint32_t b, uint32_t i, float2 v) const {
        const Split2 s = split2(v.x, v.y);
#pragma unroll
        for (int j = 0; j < 3; j++) *(uint32_t *)(at(j, b) + i) = s.p[j];
    }
};
struct PlainRows {  // f32 weights
    float *p;
    uint32_t k, rows;
    static constexpr size_t bytes(size_t rows, size_t k) { return rows * (k + 4) * 4; }
    __device__ float *at(int, uint32_t b) const { return p + b * (k + 4); }
    __device__ void put(uint32_t b, uint32_t i, float v) const { at(0, b)[i] = v; }
    __device__ void put4(uint32_t b, uint32_t i, const float4_t &v) const { *(float4_t *)(at(0, b) + i) = v; }
};
// What the two weight types do differently.  bf16: 64 k per 128 bytes of a row, activations in three pieces; f32: 32 k,
// four 16x16x4 products per 16-byte piece.
template <bool BF16> struct MfmaType;
template <> struct MfmaType<true> {
    typedef uint16_t W;
    typedef SplitRows Rows;
    static constexpr uint32_t KU = 64;
    static constexpr int PIECES = 3, XROWS = 4;  // rows of x that a wave request covers
    struct Frag { uint4 p[3]; };
    static __device__ __forceinline__ float4_t mul(const uint4 &w, const Frag &x, float4_t acc) {
        union { uint4 u; bf16x8_t v; } uw, ux;
        uw.u = w;
#pragma unroll
        for (int i = 2; i >= 0; i--) {
            ux.u = x.p[i];
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uw.v, ux.v, acc, 0, 0, 0);
        }
        return acc;
    }
};
template <> struct MfmaType<false> {
    typedef float W;
    typedef PlainRows Rows;
    static constexpr uint32_t KU = 32;
    static constexpr int PIECES = 1, XROWS = 8;
    struct Frag { uint4 p[1]; };
    static __device__ __forceinline__ float4_t mul(const uint4 &w, const Frag &x, float4_t acc) {
        union { uint4 u; float4_t v; } uw, ux;
        uw.u = w;
        ux.u = x.p[0];
        return mfma4(uw.v, ux.v, acc);
    }
    static __device__ __forceinline__ void mul(const uint4 &w, const Frag &x, float4_t &a, float4_t &b) {
        union { uint4 u; float4_t v; } uw, ux;
        uw.u = w;
        ux.u = x.p[0];
        a = __builtin_amdgcn_mfma_f32_16x16x4f32(uw.v[0], ux.v[0], a, 0, 0, 0);
        b = __builtin_amdgcn_mfma_f32_16x16x4f32(uw.v[1], ux.v[1], b, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_16x16x4f32(uw.v[2], ux.v[2], a, 0, 0, 0);
        b = __builtin_amdgcn_mfma_f32_16x16x4f32(uw.v[3], ux.v[3], b, 0, 0, 0);
    }
};
// bf16 weights and rows of activations that are bf16 already (prompts)
struct MfmaRows16 : MfmaType<true> {
    static constexpr int PIECES = 1, XROWS = 8;
    struct Frag { uint4 p[1]; };
    static __device__ __forceinline__ float4_t mul(const uint4 &w, const Frag &x, float4_t acc) {
        union { uint4 u; bf16x8_t v; } uw, ux;
        uw.u = w;
        ux.u = x.p[0];
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(uw.v, ux.v, acc, 0, 0, 0);
    }
};
// uint4 of a wave's corner: 16 weight rows x 128 bytes; per request of x its rows' KU values in pieces
template <bool BF16, bool X16 = false>
static constexpr uint32_t mfma_wave_lds(int xq) { return 128 + (BF16 && !X16 ? 96 : 64) * xq; }
// X16: x is rows of bf16, ldx elements apart
template <bool BF16, int PD, bool KEEP, int XQ, int TS, bool FOLD, bool X16, class Stage>
__device__ __forceinline__ void mfma_rows(const typename MfmaType<BF16>::W *__restrict__ w, const void *__restrict__ xp, uint64_t ldx, uint32_t k,
                                          uint32_t n, uint32_t batch, uint32_t nw, uint32_t grid, const EpiArgs &e, uint4 *lds,
                                          const typename MfmaType<BF16>::Rows &xs, Stage stage) {
    typedef std::conditional_t<X16, MfmaRows16, MfmaType<BF16>> MT;
    typedef std::conditional_t<X16, uint16_t, float> X;
    typedef typename MT::W W;
    const X *__restrict__ x = (const X *)xp;
    typedef typename MT::Frag Frag;
    constexpr uint32_t KU = MT::KU, EPP = KU / 8;  // k per pair, elements per 16-byte piece
    constexpr int XR = MT::XROWS, XN = XQ ? XQ : 1;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    static_assert(TS == 1 || XQ == 16 / XR, "parts of k need all sixteen columns");
    constexpr uint32_t R = 16 / TS;  // weight rows of a tile, activation rows of a part
    const uint32_t c = lane & 15, g = lane >> 4, cb = TS > 1 ? c : min(c, batch - 1);
    const uint32_t pairs = k / (KU * TS), pb = pairs * wave / nw, np = pairs * (wave + 1) / nw - pb, groups = (np + PD - 1) / PD;
    const uint32_t tiles = (n + R - 1) / R;
    uint4 *wl = lds + wave * mfma_wave_lds<BF16, X16>(XQ), *xl = wl + 128;
    // (a pair behind the wave's share is the share's last one again: no branches around the requests)
    auto pair_at = [&](uint32_t i) { return min(i, np - 1) * (KU * TS); };
    struct WRows { const W *p[2]; };
    auto tile_rows = [&](uint32_t tile) {
        WRows r;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t line = 8 * q + (lane >> 3);
            r.p[q] = w + (uint64_t)min(tile * R + (TS > 1 ? line % R : line), n - 1) * k + (TS > 1 ? pb * TS + line / R : pb) * KU + (lane & 7) * EPP;
        }
        return r;
    };
    const X *xr[XN];
    uint4 wr[PD][2];
    u32x4_t xv[XQ ? PD : 1][XN];  // (arrays of the struct type would be copied through scratch memory)
    auto x_request = [&](int s, uint32_t i) {
#pragma unroll
        for (int q = 0; q < XQ; q++) xv[s][q] = *(const u32x4_t *)(xr[q] + pair_at(i));
    };
    auto w_request = [&](int s, const WRows &r, uint32_t i) {
#pragma unroll
        for (int q = 0; q < 2; q++) wr[s][q] = load_stream((const uint4 *)(r.p[q] + pair_at(i)));
    };
    // 16-byte pieces of a row change places with the row, so that neither side's lanes share banks
    auto x_put = [&](int s) {
#pragma unroll
        for (int q = 0; q < XQ; q++) {
            const u32x4_t v = xv[s][q];
            if constexpr (BF16 && !X16) {
                const uint32_t r = 4 * q + (lane >> 4), at = (r * 8 + (((lane & 15) >> 1) ^ ((r >> 1) & 7))) * 2 + (lane & 1);
                const Split2 lo = split2(__uint_as_float(v.x), __uint_as_float(v.y)), hi = split2(__uint_as_float(v.z), __uint_as_float(v.w));
#pragma unroll
                for (int i = 0; i < 3; i++) *((uint2 *)(xl + i * 32 * XQ) + at) = make_uint2(lo.p[i], hi.p[i]);
            } else {
                const uint32_t r = 8 * q + (lane >> 3);
                *(u32x4_t *)(xl + r * 8 + ((lane & 7) ^ ((r >> 1) & 7))) = v;
            }
        }
    };
    auto w_put = [&](int s) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t r = 8 * q + (lane >> 3);
            wl[r * 8 + ((lane & 7) ^ (r >> 1))] = wr[s][q];
        }
    };
    auto x_get = [&](uint32_t i, int h) {  // half h of pair i
        Frag f;
#pragma unroll
        for (int j = 0; j < MT::PIECES; j++)
            f.p[j] = XQ ? xl[j * 8 * XR * XN + cb * 8 + ((4 * h + g) ^ (cb >> 1))]
                        : *(const uint4 *)(xs.at(j, cb) + pb * KU + pair_at(i) + (4 * h + g) * EPP);
        return f;
    };
    if (XQ) {
        constexpr uint32_t LPR = 64 / XR;  // lanes per row
#pragma unroll
        for (int q = 0; q < XQ; q++) {
            const uint32_t line = XR * q + lane / LPR;
            xr[q] = x + (uint64_t)min(TS > 1 ? line % R : line, batch - 1) * (X16 ? ldx : k) + (TS > 1 ? pb * TS + line / R : pb) * KU + (lane % LPR) * (16 / sizeof(X));
        }
    }
    uint32_t tile = blockIdx.x, gi = 0;
    WRows wp = tile_rows(tile);
    // Loads return in order.  Activations that stay in registers go first: they are split while the weights travel.
    // Else the order is the loop's: in any other one a wait of the loop would be for the fewest requests that either
    // order leaves behind the awaited one.
    if (XQ && KEEP) {
#pragma unroll
        for (int s = 0; s < PD; s++) x_request(s, s);
    }
#pragma unroll
    for (int s = 0; s < PD; s++) {
        if (XQ && !KEEP) x_request(s, s);
        w_request(s, wp, s);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!XQ) stage();
    Frag kept[KEEP ? PD : 1][2];
    if (KEEP) {
#pragma unroll
        for (int s = 0; s < PD; s++) {
            x_put(s);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int h = 0; h < 2; h++) kept[KEEP ? s : 0][h] = x_get(s, h);
            __builtin_amdgcn_wave_barrier();
        }
    }
    // Every second pair adds up in accumulators of its own, f32's halves of one too, so that few waves' sums are no longer than many's: not
    // shares of two pairs, unless of bf16 in two parts (8 rows of 2560 x 12352, whose waves would have one sum of twice the products they have
    // in one part: error to 64 bits 1.1e-7 in one part, 1.24e-7 with one sum, 9.9e-8 so), and not where sixteen rows of bf16 leave no registers.  f32 in four parts: the quarters of both pairs, which
    // makes two or three rows as exact as a wave per row (768 x 768, error to that form's 1.04 with halves, 0.94 so; 1.6 with one).  A pair of bf16
    // a wave (PD 1, short rows behind a norm): its halves, 9.2e-8 at 768 and 9.0e-8 at 512 (one sum 1.03e-7 and 1.01e-7, a wave per row 1.09e-7 and 9.9e-8).
    static_assert(PD > 1 || (BF16 && KEEP), "one pair a wave: short rows of bf16");
    constexpr int AS = (KEEP && (BF16 ? TS != 2 : TS < 4)) || (BF16 && XQ == 4 && TS == 1) ? 1 : 2,
                  AH = PD == 1 ? 2 : (KEEP && TS < 4) || BF16 ? 1 : KEEP ? 4 : 2;
    // What a group of PD pairs adds up to starts anew with the next one and joins the sum of the groups, so that the chains of eight waves are no
    // longer than those of sixteen (error to 64 bits, 8 rows of bf16 11008 x 4096 with sixteen waves / eight / so: 2.0e-7 / 2.9e-7 / 1.3e-7, 4 of f32 5632 x 8192 in parts of
    // k / eight waves / so: 1.3e-7 / 2.5e-7 / 1.2e-7; 324 launches, time: f32 0.998, bf16 1.003).  bf16 only for more than four pairs a wave (2048 x 2048, 4 rows, 1.02
    // otherwise) and not where sixteen columns leave no registers.
    static_assert(!FOLD || (BF16 && !KEEP && XQ < 4), "sums in groups: bf16, several groups, registers left");
    float4_t acc[AS][AH] = {}, sum_of_groups = {};
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < AS * AH; i++) acc[i / AH][i % AH] = float4_t{0.f, 0.f, 0.f, 0.f};
    };
    auto total = [&]() {
        float4_t t[AS];
#pragma unroll
        for (int s = 0; s < AS; s++) t[s] = AH == 4 ? (acc[s][0] + acc[s][AH / 4]) + (acc[s][AH / 2] + acc[s][AH - 1]) : AH == 2 ? acc[s][0] + acc[s][AH - 1] : acc[s][0];
        return AS == 2 ? t[0] + t[AS - 1] : t[0];
    };
    auto group = [&](uint32_t i0, const WRows &next, uint32_t n0, auto request) {
        if (!BF16) clear();
#pragma unroll
        for (int s = 0; s < PD; s++) {
            // (LDS serves a wave's stores and loads in order: nothing here waits for another wave)
            if (!KEEP) x_put(s);
            w_put(s);
            __builtin_amdgcn_wave_barrier();
            if (request()) {
                if (!KEEP) x_request(s, n0 + s);
                w_request(s, next, n0 + s);
                __builtin_amdgcn_sched_barrier(0);
            }
            if ((!BF16 && s == 0) || i0 + s < np) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint4 wf = wl[c * 8 + ((4 * h + g) ^ (c >> 1))];
                    float4_t &sum = acc[s % AS][h % AH];
                    if constexpr (AH == 4) MT::mul(wf, kept[s][h], acc[s][2 * h], acc[s][2 * h + 1]);
                    else if constexpr (KEEP) sum = MT::mul(wf, kept[s][h], sum);
                    else sum = MT::mul(wf, x_get(i0 + s, h), sum);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (!BF16) sum_of_groups = KEEP ? total() : sum_of_groups + total();
    };
    for (;;) {
        const bool ends = gi + 1 == groups;
        const uint32_t ntile = ends ? tile + grid : tile, ngi = ends ? 0 : gi + 1;
        const bool more = ntile < tiles;
        if (more) {
            if (ends) wp = tile_rows(ntile);
            group(gi * PD, wp, ngi * PD, [] { return true; });
        } else {
            group(gi * PD, wp, 0, [] { return false; });
        }
        if (FOLD && !ends) {
            sum_of_groups += total();
            clear();
        }
        if (ends) {
            // lane (c, g) holds lines 4 g .. + 3 of column c; a wave's corner of LDS is free
            if (TS > 1 || c < batch) *(float4_t *)(wl + lane) = !BF16 ? sum_of_groups : FOLD ? sum_of_groups + total() : total();
            if (BF16) clear();
            sum_of_groups = float4_t{0.f, 0.f, 0.f, 0.f};
            lds_barrier();
            const uint32_t row = tile * R + c;
            for (uint32_t b = wave; b < batch; b += nw) {
                // lane (c, g) adds line c of every fourth wave, in the column of its part
                float sum = 0.f;
                for (uint32_t v = g; v < nw; v += 4)
                    sum += ((const float *)(lds + v * mfma_wave_lds<BF16, X16>(XQ) + (c >> 2) * 16 + (TS > 1 ? c / R * R : 0) + b))[c & 3];
                sum = xor32_sum(xor16_sum(sum));
                if (TS == 4) sum += dpp_f32<DPP_ROW_ROR4>(sum);
                if (TS >= 2) sum += dpp_f32<DPP_ROW_ROR8>(sum);
                if (epi_gated(e.act)) {
                    const float up = lane_xor1(sum);
                    if (g == 0 && (TS == 1 || c < R) && (c & 1) == 0 && row + 1 < n) epi_store_gated(e, b, row / 2, sum, up);
                } else if (g == 0 && (TS == 1 || c < R) && row < n) {
                    epi_store<true>(e, b, row, sum);
                }
            }
            if (more) lds_barrier();
        }
        if (!more) break;
        tile = ntile;
        gi = ngi;
    }
}

// The staging of a folded norm for mfma_rows: wave b normalises row b (every row in front of a norm over all) in its registers (16 bytes of every 256 elements a
// lane, k <= 256 VM) and puts it into LDS split.  stage_normed_rows spreads every row over all waves, a trip through
// LDS and a barrier for each of two sums and a chain of 16 reads behind them: 13.9 us for a folded launch of 8 rows of
// 768 x 2304 in f32, whose product alone takes 4.3.
template <int NORM, int VM, class Rows>
__device__ __forceinline__ void stage_rows_by_wave(float *sh, const float *__restrict__ x, uint32_t k, uint32_t batch,
                                                   const float *__restrict__ nscale, const float *__restrict__ nbias, float eps,
                                                   uint64_t ldx, const PostNorm &post, const Rows &xs, uint32_t b) {
    const uint32_t lane = threadIdx.x & 63, n4 = k / 4;
    const bool on = b < batch;
    const float *row = NORM == 3 ? post.y + (uint64_t)b * k : x + (uint64_t)b * ldx;
    auto row_sum = [](float t) { return xor32_sum(xor16_sum(group_sum<16>(t))); };
    // (Sums in f64 next to a long row and its scale would spill.  Rows that long are at most eight, so that the last wave,
    // which has none, brings the scale into LDS.)
    constexpr bool SCALE_LDS = NORM == 4 && VM == 8, BIAS = (NORM == 1 || NORM == 4) && VM == 4;  // (the bias of a short row comes with it)
    float *gs = sh + 64;
    float4_t v[VM], g[SCALE_LDS ? 1 : VM], bias[BIAS ? VM : 1];
    if (on) {
        if constexpr (BIAS) {
            const float *nb = nbias ? nbias : nscale;
#pragma unroll
            for (int u = 0; u < VM; u++) bias[u] = *(const float4_t *)(nb + 4 * min(lane + 64 * u, n4 - 1));
        }
#pragma unroll
        for (int u = 0; u < VM; u++) v[u] = *(const float4_t *)(row + 4 * min(lane + 64 * u, n4 - 1));
        if constexpr (!SCALE_LDS) {
#pragma unroll
            for (int u = 0; u < VM; u++) g[u] = *(const float4_t *)(nscale + 4 * min(lane + 64 * u, n4 - 1));
        }
    } else if (SCALE_LDS && b == 15) {
#pragma unroll
        for (int u = 0; u < VM; u++)
            if (lane + 64 * u < n4) *(float4_t *)(gs + 4 * (lane + 64 * u)) = *(const float4_t *)(nscale + 4 * (lane + 64 * u));
    }
    float mean = 0.f, rs;
    if constexpr (NORM == 4) {
        // Whole slice: sums of x - x[0] and of its square in f64, one trip through LDS (norm_sequence_part_kernel's, which serves the
        // longer prompts).
        double *shd = (double *)sh, sum = 0.0, sq = 0.0;
        const double ref = x[0];
        if (on) {
#pragma unroll
            for (int u = 0; u < VM; u++) {
                if (lane + 64 * u < n4)
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const double d = v[u][t] - ref;
                        sum += d;
                        sq = fma(d, d, sq);
                    }
                __builtin_amdgcn_sched_barrier(0);  // (converted all at once, the row spills)
            }
            sum = wave_sum_f64(sum);
            sq = wave_sum_f64(sq);
            if (lane == 0) { shd[b] = sum; shd[16 + b] = sq; }
        }
        __syncthreads();
        if (!on) return;
        const double inv = inv_count(k * batch), off = wave_sum_f64(lane < batch ? shd[lane] : 0.0) * inv;
        mean = (float)(ref + off);
        rs = whole_norm_rs(fma(-off, off, wave_sum_f64(lane < batch ? shd[16 + lane] : 0.0) * inv), eps);
    } else {
        if (!on) return;
        if (NORM == 1) {
            float sum = 0.f;
#pragma unroll
            for (int u = 0; u < VM; u++) sum += lane + 64 * u < n4 ? (v[u][0] + v[u][1]) + (v[u][2] + v[u][3]) : 0.f;
            mean = row_sum(sum) / (float)k;
        }
        float sq = 0.f;
#pragma unroll
        for (int u = 0; u < VM; u++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float d = lane + 64 * u < n4 ? v[u][t] - mean : 0.f;
                sq = fmaf(d, d, sq);
            }
        rs = 1.0f / sqrtf(row_sum(sq) / (float)k + eps);
    }
#pragma unroll
    for (int u = 0; u < VM; u++) {
        const uint32_t i = 4 * (lane + 64 * u);
        if (i >= k) continue;
        float4_t o, gu;
        if constexpr (SCALE_LDS) gu = *(const float4_t *)(gs + i);
        else gu = g[u];
        if (NORM == 3) {
            const float4_t h = *(const float4_t *)(x + (uint64_t)b * ldx + i);
            float4_t ls = {1.f, 1.f, 1.f, 1.f};
            if (post.ls) ls = *(const float4_t *)(post.ls + i);
#pragma unroll
            for (int t = 0; t < 4; t++) o[t] = fmaf(v[u][t] * rs * gu[t], ls[t], h[t]);
            if (blockIdx.x == 0) *(float4_t *)(post.h_out + (uint64_t)b * k + i) = o;
        } else {
            float4_t bi = {0.f, 0.f, 0.f, 0.f};
            if constexpr (BIAS) { if (nbias) bi = bias[u]; }
            else if (NORM != 2 && nbias) bi = *(const float4_t *)(nbias + i);
#pragma unroll
            for (int t = 0; t < 4; t++) o[t] = gu[t] * (v[u][t] - mean) * rs + bi[t];
        }
        xs.put4(b, i, o);
    }
}

static constexpr size_t kDenseNormLdsLimit = 64 * 1024;
// rows + scale + bias + per-wave partial sums + statistics
static constexpr size_t gemv_dense_norm_lds(uint64_t k, uint32_t bp) { return ((size_t)(bp + 2) * k + 16 * bp + 32) * 4; }
static constexpr size_t gemv_dense_post_lds(uint64_t k, uint32_t bp) { return gemv_dense_norm_lds(k, bp) + (size_t)bp * k * 4; }
// The most pairs of chunks in a row that a folded norm over bp rows leaves room for, and of these in the share of one of up to 16 waves
// (f32, which is always 16 of them, 0: a wave has none).  Nothing is built for more.
template <bool BF16>
static constexpr uint32_t gemv_fold_row_pairs(int norm, uint32_t bp) {
    const uint64_t ku = MfmaType<BF16>::KU;
    uint32_t pairs = 0;
    while ((norm == 3 ? gemv_dense_post_lds((pairs + 1) * ku, bp) : gemv_dense_norm_lds((pairs + 1) * ku, bp)) <= kDenseNormLdsLimit) pairs++;
    return pairs;
}
template <bool BF16>
static constexpr uint32_t gemv_fold_share(int norm, uint32_t bp) {
    const uint32_t pairs = gemv_fold_row_pairs<BF16>(norm, bp);
    return BF16 || pairs >= 16 ? (pairs + 15) / 16 : 0;
}

// NORM 0: BP rows (padded to 4, 8 or 16) in global memory; else staged normalised in LDS behind the waves' corners.
template <bool BF16, int BP, int NORM, int PD, bool KEEP, int TS = 1, bool FOLD = false, bool X16 = false>
__global__ __launch_bounds__(1024) void gemv_mfma_kernel(const typename MfmaType<BF16>::W *__restrict__ w, const float *__restrict__ x, uint32_t k,
                                                         uint32_t n, uint32_t batch, uint32_t waves, uint32_t grid, EpiArgs e,
                                                         const float *__restrict__ nscale, const float *__restrict__ nbias, float eps,
                                                         uint64_t ldx, PostNorm post) {
    extern __shared__ uint4 mlds[];
    typedef typename MfmaType<BF16>::Rows Rows;
    constexpr int XROWS = X16 ? MfmaRows16::XROWS : MfmaType<BF16>::XROWS, XQ = NORM ? 0 : ((TS > 1 ? 16 : BP) + XROWS - 1) / XROWS;
    // a folded norm: the split rows first; what its staging needs lies where the corners will be
    const Rows xs{(decltype(Rows::p))mlds, k, (uint32_t)BP};
    uint4 *corners = NORM ? (uint4 *)((char *)mlds + Rows::bytes(BP, k)) : mlds;
    mfma_rows<BF16, PD, KEEP, XQ, TS, FOLD, X16>(w, x, ldx, k, n, batch, waves, grid, e, corners, xs, [&]() {
        if constexpr (NORM != 0) {
            constexpr uint32_t LONGEST = gemv_fold_row_pairs<BF16>(NORM, BP) * MfmaType<BF16>::KU;
            const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            if (LONGEST <= 1024 || k <= 1024) {
                stage_rows_by_wave<NORM, 4>((float *)corners, x, k, batch, nscale, nbias, eps, ldx, post, xs, wave);
                // (a pair a wave: there may be more rows than waves)
                if constexpr (PD == 1 && NORM != 4)
                    for (uint32_t b = wave + waves; b < batch; b += waves)
                        stage_rows_by_wave<NORM, 4>((float *)corners, x, k, batch, nscale, nbias, eps, ldx, post, xs, b);
            } else if (LONGEST <= 2048 || k <= 2048) stage_rows_by_wave<NORM, 8>((float *)corners, x, k, batch, nscale, nbias, eps, ldx, post, xs, wave);
            else
                stage_normed_rows<BP, NORM>((float *)corners, x, k, batch, nscale, nbias, eps, ldx, post,
                                            [&](uint32_t b, uint32_t i, float v) { xs.put(b, i, v); });
            __syncthreads();
        }
    });
}

// (a norm over all rows: the partial sums in f64)
static size_t gemv_whole_norm_lds(uint64_t k, uint32_t bp) { return gemv_dense_norm_lds(k, bp) + (size_t)16 * bp * 4; }

// True when the dense decode matmul can take the normalisation into its staging: the normalised
// activation block [batch padded, k] f32 has to fit in LDS.
bool gemv_can_fuse_norm_dense(const Weight &w, uint64_t batch) {
    if (w.dtype >= COEUS_W_Q8_0 || batch < 1 || batch > 16) return false;
    return gemv_dense_norm_lds(w.k, pad_batch(batch)) <= kDenseNormLdsLimit;
}

// Weights whose rows are whole pairs of chunks (128 bytes), one for every wave at least, and none of whose values is infinite
// (an activation's three bf16 may be zero).
static bool gemv_mfma_shape(const Weight &w, uint32_t waves) {
    const uint64_t ku = w.dtype == COEUS_W_BF16 ? 64 : 32;
    return w.dtype <= COEUS_W_BF16 && !w.infinite && w.k % ku == 0 && w.k / ku >= waves && w.k < (1ull << 31) && w.n < (1ull << 31) - 16;
}
// Where the matrix cores are the faster of the two (us with weights from memory: a wave per row / here).
static bool gemv_uses_mfma(const Weight &w, uint64_t batch, uint32_t waves, bool folded) {
    if (!gemv_mfma_shape(w, waves) || batch < 1) return false;
    const bool bf = w.dtype == COEUS_W_BF16;
    // One row (two weight rows a wave / here): short rows of which there are many (256 x 16384 5.0 / 4.4, x 100000 18.3 / 11.1, 512 x 50257 12.6 / 10.8;
    // but 512 x 12000 0.89 of the time, 576 x 50257 0.89), and long ones a little beyond the 2048 that give every compute unit one
    // workgroup (11008 x 3072 17.7 / 16.8, 14336 x 3072 20.6 / 19.0 with sixteen waves, 0.94 and 0.96 of that with eight; x 2048 0.74 of the time, x 3584 the
    // same, 8192 x 3072 the same).
    if (batch == 1) return bf && !folded && (w.k <= 512 ? w.n >= 16384 : w.k >= 10240 && w.n > 2048 && w.n <= 3328);
    // (A norm in front costs a wave per row more: f32, 2 rows of 768 x 768 7.4 / 5.8.  Two rows of bf16 are the exception where they
    // are long and few: 2560 x 4096 11.0 / 11.6, x 12288 22.7 / 19.1.)
    if (folded) return !(bf && batch == 2 && w.k > 2048 && w.n <= 4096);
    // Two or three rows on few tiles: a wave per row keeps more compute units busy, unless the tiles are dealt in parts of k (f32 up to 1024 outputs, with
    // sums as near to 64 bits: 3 rows of 768 x 768 4.3 / 3.6, 8192 x 1024 16.6 / 8.6).  f32, 2 rows of
    // 1024 x 1536 4.4 / 4.7, but 1024 x 2304 5.2 / 5.1, 2048 x 1152 6.5 / 6.2; 3 rows of 1024 x
    // 1152 4.9 / 4.6; bf16, 2 rows of 1024 x 256 3.2 / 3.4, but x 1280 3.5 / 3.5, 1536 x 256 4.0 / 3.8.
    if (!bf && batch <= 3) return w.k <= 256 || (w.n <= 1024 ? w.k % 128 == 0 : batch == 3 || w.k > 1024 || w.n > 2048);
    if (bf && batch == 2) return w.k <= 256 || w.k > 1024 || w.n > 1024;
    return true;
}
// Waves of a plain launch: as many as have two pairs of chunks each.
static uint32_t gemv_mfma_waves(uint64_t pairs) { return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(16, (pairs + 1) / 2)); }
bool gemv_takes_f32_rows(const Weight &w, uint64_t rows) {
    return w.dtype == COEUS_W_F32 && rows >= 2 && rows <= 16 && gemv_mfma_shape(w, gemv_mfma_waves(w.k / 32));
}
// Waves behind a folded norm: sixteen, or one for each pair of a shorter row of bf16.  Those took the kernel with a wave per output row, whose
// workgroups convert every row again for each of them.  Decode steps of 12 layers of 768, ms, that one / the norm a launch of its own / this: 2, 4, 8 and
// 16 rows 0.42 / 0.46 / 0.38, 0.50 / 0.46 / 0.38, 0.72 / 0.50 / 0.43, 1.19 / 0.62 / 0.56; of 512 0.41 / 0.44 / 0.37, 0.48 / 0.45 / 0.39, 0.66 / 0.47 / 0.40,
// 1.08 / 0.56 / 0.49.  (f32 below 512 stays: sums of pairs, even in quarters, are 1 % less exact than a wave per row's.)
static uint32_t gemv_fold_waves(const Weight &w) { return w.dtype == COEUS_W_BF16 ? (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(16, w.k / 64)) : 16; }
static size_t gemv_mfma_norm_lds(const Weight &w, uint32_t bp, size_t staging) {
    const bool bf = w.dtype == COEUS_W_BF16;
    return (bf ? SplitRows::bytes(bp, w.k) : PlainRows::bytes(bp, w.k)) + std::max((size_t)16 * 16 * 128, staging);
}
static bool gemv_folds_on_mfma(const Weight &w, uint64_t batch, size_t staging) {
    const uint32_t waves = gemv_fold_waves(w);
    return gemv_uses_mfma(w, batch, waves, true) && gemv_mfma_norm_lds(w, pad_batch(batch), staging) <= 160 * 1024;
}
bool gemv_can_fuse_whole_norm(const Weight &w, uint64_t batch) {
    if (w.dtype != COEUS_W_F32 || batch < 2 || batch > 16 || !gemv_can_fuse_norm_dense(w, batch) || !gemv_uses_mfma(w, batch, 16, true)) return false;
    const uint32_t bp = pad_batch(batch);
    return gemv_mfma_norm_lds(w, bp, gemv_whole_norm_lds(w.k, bp)) <= 160 * 1024;
}
bool gemv_can_fuse_post_norm(const Weight &w, uint64_t batch) {
    if (w.dtype >= COEUS_W_Q8_0 || batch < 1 || batch > 16) return false;
    return gemv_dense_post_lds(w.k, pad_batch(batch)) <= kDenseNormLdsLimit;
}

// ---------------------------------------------------------------- dense kernel behind hyper-connections
// x holds `streams` rows per batch entry, y the output of the sublayer before.  A workgroup stages the layer norm
// of sum_t in[t] x'_t, x'_t = sum_s mix[s][t] x_s + mult out[t] y, and multiplies its rows of the weight with it; the
// first workgroup stores the x'_t.  What a sum over t needs of the old streams is one coefficient per stream
// (hyper_fold_kernel), so only that workgroup forms the new ones.
//
// Five rows of f32 in front of every share of the weight are what this costs, and a compute unit's trips to memory
// bound it: one workgroup of 16 waves per compute unit reads them once and then every rows-th row of the weight,
// with SL steps in flight across the rows' ends.  The activation rows pass through registers (pairs of elements,
// NIT per thread): a wave finds the mean and the squares about it of its own elements, and one barrier later every
// wave merges the sixteen of them.  What the first loads need lies in the 64 bytes of arguments that arrive with
// the wave.
constexpr int kFusedStreams = (int)kMaxFoldedStreams;
// what x_s [4] and y contribute to the weighted sum of the new streams, mult out[t] [4], mix [4][4]; zeros behind
// the streams there are
struct HyperFold {
    float cs[kFusedStreams], om[kFusedStreams], mix[kFusedStreams][kFusedStreams], cy;
};
static_assert(sizeof(HyperFold) <= kHyperFoldFloats * 4, "size of a record");

__global__ __launch_bounds__(64) void hyper_fold_kernel(const float *mix, const float *out, const float *in, float mult, uint32_t S,
                                                        HyperFold *f) {
    const uint32_t t = threadIdx.x;
    if (t < 16) f->mix[t / 4][t % 4] = mix && t / 4 < S && t % 4 < S ? mix[t / 4 * S + t % 4] : 0.f;
    if (t < 4) {
        f->om[t] = out && t < S ? mult * out[t] : 0.f;
        float c = 0.f;
        if (t < S) {
            if (!mix) c = in[t];
            else for (uint32_t u = 0; u < S; u++) c = fmaf(mix[t * S + u], in[u], c);
        }
        f->cs[t] = c;
    }
    if (t == 0) {
        float c = 0.f;
        if (out)
            for (uint32_t u = 0; u < S; u++) c = fmaf(mult * out[u], in[u], c);
        f->cy = c;
    }
}

int launch_hyper_fold(const float *mix, const float *out, const float *in, float mult, uint32_t streams, float *fold, hipStream_t st) {
    if (!in || !fold || !mix != !out || streams < 1 || streams > kFusedStreams)
        return fail(COEUS_INVALID_INPUT, "folded hyper-connections: bad arguments or too many streams");
    hipLaunchKernelGGL(hyper_fold_kernel, dim3(1), dim3(64), 0, st, mix, out, in, mult, streams, (HyperFold *)fold);
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

template <bool BF16, int BP, int NIT, bool MF = false>
__global__ __launch_bounds__(1024) void gemv_hyper_kernel(const void *__restrict__ wdata, const float *__restrict__ x,
                                                          const float *__restrict__ y, const float *__restrict__ norm,
                                                          const HyperFold *__restrict__ fold, uint32_t k, uint32_t batch_streams,
                                                          float *x_out, float eps, EpiArgs e) {
    constexpr int NS = kFusedStreams, SL = 4;
    // [BP][k]; MF: the waves' corners (mfma_rows), the rows' pieces
    extern __shared__ __attribute__((aligned(16))) float hyper_lds[];
    float *xn = MF ? hyper_lds + 16 * 4 * mfma_wave_lds<true>(0) : hyper_lds;
    __shared__ float2 red[16][BP];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), S = batch_streams >> 16,
                   batch = batch_streams & 0xffffu;
    const bool vec = (k & 7) == 0, gated = epi_gated(e.act);
    // Unit u of this wave (a row, or the two rows of a gated pair) is unit blockIdx.x + gridDim.x (wave + 16 u) of
    // the weight.
    const uint32_t per = gated ? 2 : 1, units = (uint32_t)(e.n / per), first = blockIdx.x + gridDim.x * wave, stride = 16 * gridDim.x;
    const uint32_t rows = first < units ? ((units - 1 - first) / stride + 1) * per : 0, steps = (k + 511) / 512, items = rows * steps;
    auto row_of = [&](uint32_t i) { return gated ? 2ull * (first + stride * (i >> 1)) + (i & 1) : (uint64_t)first + (uint64_t)stride * i; };
    // item t: step t % steps of row t / steps; a lane behind the row's end re-reads the last weights
    uint32_t ld_row = 0, ld_step = 0;
    auto wload = [&](uint4 &a, uint4 &b) {
        if (ld_row >= rows) return;
        constexpr uint32_t ES = BF16 ? 2 : 4;
        const char *base = (const char *)wdata + row_of(ld_row) * k * ES;  // wave-uniform
        const uint32_t off = min(lane * 8 + 512 * ld_step, k - 8) * ES;
        if (++ld_step == steps) { ld_step = 0; ld_row++; }
        a = load_stream((const uint4 *)(base + off));
        if (!BF16) b = load_stream((const uint4 *)(base + off + 16));
    };
    // Where element i of the normalised rows lies: the two quads of every eight in halves of their own, so that the
    // lanes of a read of quads are neighbours.
    // (MF: split, as mfma_rows takes them)
    const SplitRows xs{(uint16_t *)xn, k, (uint32_t)BP};
    auto place = [&](uint32_t i) { return vec ? (i & 4 ? k / 2 : 0) + (i >> 3) * 4 + (i & 3) : i; };
    // The streams are requested before the weights: loads return in order, and the norm needs only the streams.
    // (No branches here: a lane behind the end re-reads the last elements, a stream that is not there the last one.)
    float2 xv[NIT][BP][NS], yv[NIT][BP], g[NIT];
#pragma unroll
    for (int it = 0; it < NIT; it++) {
        const uint32_t i = min(2 * (tid + 1024 * it), k - 2);
        g[it] = *(const float2 *)(norm + i);
#pragma unroll
        for (int b = 0; b < BP; b++) {
            const uint32_t row = min((uint32_t)b, batch - 1);
#pragma unroll
            for (int s = 0; s < NS; s++) xv[it][b][s] = *(const float2 *)(x + ((uint64_t)row * S + min((uint32_t)s, S - 1)) * k + i);
            yv[it][b] = *(const float2 *)(y + (uint64_t)row * k + i);
        }
    }
    auto row_sum = [](float t) { return xor32_sum(xor16_sum(group_sum<16>(t))); };
    auto normalise = [&]() {
        float2 v[NIT][BP];
        float cnt = 0.f;  // elements of this wave
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const uint32_t i = 2 * (tid + 1024 * it), w0 = 2 * (64 * wave + 1024 * it);
            cnt += w0 < k ? (float)min(128u, k - w0) : 0.f;
#pragma unroll
            for (int b = 0; b < BP; b++) {
                float2 o = make_float2(fold->cy * yv[it][b].x, fold->cy * yv[it][b].y);
#pragma unroll
                for (int s = 0; s < NS; s++) { o.x = fmaf(fold->cs[s], xv[it][b][s].x, o.x); o.y = fmaf(fold->cs[s], xv[it][b][s].y, o.y); }
                v[it][b] = i < k ? o : make_float2(0.f, 0.f);
            }
        }
        if (blockIdx.x == 0 && x_out) {
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                const uint32_t i = 2 * (tid + 1024 * it);
#pragma unroll
                for (int b = 0; b < BP; b++) {
                    if (b >= (int)batch || i >= k) continue;
#pragma unroll
                    for (int u = 0; u < NS; u++) {
                        if (u >= (int)S) continue;
                        float2 nv = make_float2(fold->om[u] * yv[it][b].x, fold->om[u] * yv[it][b].y);
#pragma unroll
                        for (int s = 0; s < NS; s++) {
                            nv.x = fmaf(fold->mix[s][u], xv[it][b][s].x, nv.x);
                            nv.y = fmaf(fold->mix[s][u], xv[it][b][s].y, nv.y);
                        }
                        *(float2 *)(x_out + ((uint64_t)b * S + u) * k + i) = nv;
                    }
                }
            }
        }
        const float inv_cnt = cnt > 0.f ? 1.0f / cnt : 0.f;
#pragma unroll
        for (int b = 0; b < BP; b++) {
            if (b >= (int)batch) continue;
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int it = 0; it < NIT; it++) s1 += v[it][b].x + v[it][b].y;
            const float own = row_sum(s1), mw = own * inv_cnt;
#pragma unroll
            for (int it = 0; it < NIT; it++)
                if (2 * (tid + 1024 * it) < k) {
                    const float dx = v[it][b].x - mw, dy = v[it][b].y - mw;
                    s2 = fmaf(dx, dx, s2); s2 = fmaf(dy, dy, s2);
                }
            s2 = row_sum(s2);
            if (lane == 0) red[wave][b] = make_float2(own, s2);
        }
        __syncthreads();
        {
            // lane w of 16 takes wave w's record
            const uint32_t w = lane & 15;
            float cw = 0.f;
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                const uint32_t w0 = 2 * (64 * w + 1024 * it);
                cw += w0 < k ? (float)min(128u, k - w0) : 0.f;
            }
#pragma unroll
            for (int b = 0; b < BP; b++) {
                if (b >= (int)batch) continue;
                const float2 rec = red[w][b];
                const float mean = group_sum<16>(rec.x) / (float)k, dm = cw > 0.f ? rec.x / cw - mean : 0.f;
                const float rs = 1.0f / sqrtf(group_sum<16>(fmaf(cw * dm, dm, rec.y)) / (float)k + eps);
#pragma unroll
                for (int it = 0; it < NIT; it++) {
                    const uint32_t i = 2 * (tid + 1024 * it);
                    const float2 o = make_float2((v[it][b].x - mean) * rs * g[it].x, (v[it][b].y - mean) * rs * g[it].y);
                    if (i < k) {
                        if (MF) xs.put2(b, i, o);
                        else *(float2 *)(xn + (size_t)b * k + place(i)) = o;
                    }
                }
            }
        }
        __syncthreads();
    };
    if constexpr (MF) {
        __builtin_amdgcn_sched_barrier(0);
        mfma_rows<true, 2, true, 0, 1, false, false>((const uint16_t *)wdata, nullptr, k, k, (uint32_t)e.n, batch, 16, gridDim.x, e, (uint4 *)hyper_lds, xs, [&]() {
            __builtin_amdgcn_sched_barrier(0);
            normalise();
        });
        return;
    }
    __builtin_amdgcn_sched_barrier(0);
    uint4 wa[SL], wb[SL];
#pragma unroll
    for (int q = 0; q < SL; q++) {
        wa[q] = wb[q] = make_uint4(0, 0, 0, 0);
        if (vec) wload(wa[q], wb[q]);
    }
    __builtin_amdgcn_sched_barrier(0);
    normalise();
    float acc[BP], gate[BP];
#pragma unroll
    for (int b = 0; b < BP; b++) acc[b] = gate[b] = 0.f;
    // a row is complete: its epilogue (the first row of a pair only keeps its sums)
    auto finish = [&](uint32_t i) {
#pragma unroll
        for (int b = 0; b < BP; b++) {
            const float sum = row_sum(acc[b]);
            acc[b] = 0.f;
            if (gated && (i & 1) == 0) { gate[b] = sum; continue; }
            if (lane != 0 || b >= (int)batch) continue;
            if (gated) epi_store_gated(e, b, row_of(i) / 2, gate[b], sum);
            else epi_store<true>(e, b, row_of(i), sum);
        }
    };
    if (vec) {
        uint32_t row = 0, step = 0;
        for (uint32_t t = 0; t < items; t += SL)
#pragma unroll
            for (int q = 0; q < SL; q++) {
                if (t + q >= items) break;  // wave-uniform
                const uint32_t k0 = lane * 8 + 512 * step;
                if (k0 < k) {
                    float wv[8];
                    if (BF16) {
                        const uint32_t r[4] = {wa[q].x, wa[q].y, wa[q].z, wa[q].w};
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            wv[2 * j] = __uint_as_float(r[j] << 16);
                            wv[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u);
                        }
                    } else {
                        const uint32_t r[8] = {wa[q].x, wa[q].y, wa[q].z, wa[q].w, wb[q].x, wb[q].y, wb[q].z, wb[q].w};
#pragma unroll
                        for (int j = 0; j < 8; j++) wv[j] = __uint_as_float(r[j]);
                    }
#pragma unroll
                    for (int b = 0; b < BP; b++) {
                        if (b >= (int)batch) continue;
                        const float *xr = xn + (size_t)b * k + k0 / 2;
                        const float4 xa = *(const float4 *)xr, xb = *(const float4 *)(xr + k / 2);
                        float s = acc[b];
                        s = fmaf(wv[0], xa.x, s); s = fmaf(wv[1], xa.y, s); s = fmaf(wv[2], xa.z, s); s = fmaf(wv[3], xa.w, s);
                        s = fmaf(wv[4], xb.x, s); s = fmaf(wv[5], xb.y, s); s = fmaf(wv[6], xb.z, s); s = fmaf(wv[7], xb.w, s);
                        acc[b] = s;
                    }
                }
                wload(wa[q], wb[q]);
                if (++step == steps) { finish(row); step = 0; row++; }
            }
    } else {
        for (uint32_t i = 0; i < rows; i++) {
            for (uint32_t kk = lane; kk < k; kk += 64) {
                const uint64_t at = row_of(i) * k + kk;
                const float wv = BF16 ? bf16_bits_to_f32(((const uint16_t *)wdata)[at]) : ((const float *)wdata)[at];
#pragma unroll
                for (int b = 0; b < BP; b++)
                    if (b < (int)batch) acc[b] = fmaf(wv, xn[(size_t)b * k + kk], acc[b]);
            }
            finish(i);
        }
    }
}

// pairs of elements per thread; beyond four over the batch every workgroup would read more rows than it is worth
static uint32_t hyper_pairs(uint64_t k) { return (uint32_t)ceil_div(k, 2048); }
bool gemv_can_fuse_hyper(const Weight &w, uint64_t batch, uint64_t streams) {
    if (w.dtype >= COEUS_W_Q8_0 || batch < 1 || batch > 16 || streams < 1 || streams > kFusedStreams || (w.k & 1)) return false;
    const uint32_t bp = pad_batch(batch), nit = hyper_pairs(w.k);
    return nit <= 3 && bp * nit <= 4;
}

template <bool BF16>
static int launch_gemv_hyper(const Weight &w, uint64_t batch, const EpiArgs &e, hipStream_t st, const NormFuse &nf) {
    if (!gemv_can_fuse_hyper(w, batch, nf.streams) || !nf.h || !nf.scale || !nf.fold || nf.kind != COEUS_NORM_LAYERNORM || nf.ld ||
        nf.bias || (nf.y && (!nf.h_out || nf.h_out == nf.h)))
        return fail(COEUS_INVALID_INPUT, "folded hyper-connections: bad arguments or too many streams");
    const uint32_t bp = pad_batch(batch), b = (uint32_t)batch, k = (uint32_t)w.k, nit = hyper_pairs(w.k);
    // (the matrix-core instance lays its LDS out for two rows: one stays with a wave per weight row, and in front of three or
    // four a model's step has a launch of its own)
    const bool mf = BF16 && nit == 1 && bp == 2 && gemv_uses_mfma(w, batch, 16, true);
    const size_t lds = mf ? 16 * 16 * mfma_wave_lds<true>(0) + SplitRows::bytes(bp, k) : (size_t)bp * k * 4;  // (57 KiB at most)
    const uint32_t bs = b | nf.streams << 16;
    const HyperFold *fold = (const HyperFold *)nf.fold;
    const float *y = nf.y ? nf.y : nf.h;  // (without an output of a sublayer before its weight is zero)
    float *x_out = nf.y ? nf.h_out : nullptr;
    if (w.n > 0x7fffffffull) return fail(COEUS_INVALID_INPUT, "folded hyper-connections: too many rows");
    const uint64_t units = epi_gated(e.act) ? w.n / 2 : w.n;
    const dim3 grid((unsigned)std::min<uint64_t>(256, mf ? ceil_div(w.n, 16) : units)), block(1024);  // (a workgroup per compute unit)
    if constexpr (BF16) {
        if (mf) {
            hipLaunchKernelGGL((gemv_hyper_kernel<true, 2, 1, true>), grid, block, lds, st, w.data, nf.h, y, nf.scale, fold, k, bs, x_out, nf.eps, e);
            COEUS_HIP(hipGetLastError());
            return COEUS_OK;
        }
    }
#define COEUS_GH(BPV, NV) \
    hipLaunchKernelGGL((gemv_hyper_kernel<BF16, BPV, NV>), grid, block, lds, st, w.data, nf.h, y, nf.scale, fold, k, bs, x_out, nf.eps, e)
    if (bp == 4) COEUS_GH(4, 1);
    else if (bp == 2 && nit == 1) COEUS_GH(2, 1);
    else if (bp == 2) COEUS_GH(2, 2);
    else if (nit == 1) COEUS_GH(1, 1);
    else if (nit == 2) COEUS_GH(1, 2);
    else COEUS_GH(1, 3);
#undef COEUS_GH
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// One plain row: two weight rows a wave where that is the faster form (us, the other one / here).
// f32, against a wave per row with as many steps in flight (gemv_one_row_steps; the same bits): long rows where the 2048 that give every compute unit a
// workgroup come out nearly even, or are many times that (time over the other's: 2048 x 8192 1.00, x 16384 0.95, x 33792 0.93, 3072 x 8192 0.95, x 14336 0.91, 7168 x 4096 0.96, 2560 x
// 2048 - 25600 0.99 - 1.04; but x 2304 1.15 - 1.22, x 3600 1.00 - 1.04, x 5120 1.09 - 1.13, x 9216 1.00 - 1.05, rows a multiple of 16 KiB apart x 16384 - 32000 1.03, 1536 long 0.99 - 1.05),
// short ones of very many (768 x 50257 0.99, x 32000 1.00, x 22016 1.03; 1032 x 8192 - 50257 1.06 - 1.09).  Gated pairs, against the general form
// that holds them in two waves: from 1536 of k on beyond 3200 rows, from 1032 and 8192, and up to the 2048 that give every compute unit one workgroup, but not a little beyond
// these (1536 - 8192 x 1500 - 2048 0.85 - 1.01, x 2304 1.05 - 1.12, x 3600 0.90 - 0.97, x 22016 0.85 - 0.93, x 1024 1.01 - 1.08).  bf16: all that the matrix cores do not take (gemv_uses_mfma), but rows 32 KiB apart, which share their memory channels,
// are a wave's each between 4096 and 6144 of them (16384 x 4608 1.07, 32768 x 4608 1.14; x 6144 1.00, x 8192 0.86), and so are up
// to 8192 rows of one step, without a gate (64 - 512 x 128 - 8192 1.02 of the time in the mean, x 10000 - 16000 0.94; gated pairs of one step 0.85 - 0.97), and up to 1024 of
// more than two steps (1032 x 1030 0.99, x 768 0.98 of the time with a wave per row, 2048 x 1024 0.92, 11008 x 1024 0.80, but 1536 x 1536 1.07).
static bool gemv_takes_many(const Weight &w, uint64_t batch, bool gated = false) {
    if (batch != 1 || w.dtype > COEUS_W_BF16 || w.k % 8 || w.k >= (1ull << 31) || w.n >= (1ull << 31) - 8) return false;
    if (w.dtype == COEUS_W_BF16)
        return !gemv_uses_mfma(w, 1, gemv_mfma_waves(w.k / MfmaType<true>::KU), false) && !(w.k % 16384 == 0 && w.n > 4096 && w.n < 6144) &&
               (gated || w.k > 512 || w.n > 8192) && (gated || w.k <= 1024 || w.n > 1024);
    if (w.k >= 1536 && gated) return (w.n > 1024 && w.n <= 2048) || w.n > 3200;
    if (w.k >= 1536) return w.k >= 2048 && w.k % 4096 && (w.n >= 16384 || 12 * round_up(w.n, 2048) <= 13 * w.n);
    return w.k > 1024 ? gated && w.n >= 8192 : w.k > 512 && w.k < 1024 && w.n >= (gated ? 20000 : 32001);
}

// One plain row of the others: steps in flight of a weight row a wave (f32 1 - 4, bf16 1, 4 or 6: gemv_takes_many has bf16 rows of two steps; 0: the
// general form, for gates, whose pairs it holds in two waves, and lengths that are no multiple of 8).  f32 (us with 2 / 3 / 4 / 6): two where a workgroup a CU and less is all there is (8192 x 1024 8.98 /
// 9.18 / 9.04 / 9.43, 16384 x 768 15.1 / - / 15.6), else three or four, whichever asks for fewer steps in vain (4096 x 3072 13.1 / 13.3 / 12.8 /
// 14.7, 3072 x 3072 10.8 / 10.6 / 10.9 / 10.9).  bf16: four, or six where they are fewer trips with no more in vain (3072 x 768 3.99 / 3.50 / 3.53 / 3.39,
// 8192 x 1024 6.70 / 5.79 / 5.18 / 5.40); rows 32 KiB apart stay with the general form (16384 x 4608 30.8, two steps of these 34.2, four 32.7).
static uint32_t gemv_one_row_steps(const Weight &w, uint64_t batch, bool gated) {
    if (batch != 1 || w.dtype > COEUS_W_BF16 || w.k % 8 || w.k >= (1ull << 31) || w.n >= (1ull << 31) - 8 || gated) return 0;
    const uint64_t steps = ceil_div(w.k, 512);
    if (steps <= 2) return (uint32_t)steps;
    auto slots = [&](uint64_t d) { return ceil_div(steps, d) * d; };
    if (w.dtype == COEUS_W_F32) return w.n <= 1024 ? 2 : slots(3) < slots(4) ? 3 : 4;
    return w.n > 1024 ? 0 : slots(6) <= slots(4) && steps % 4 ? 6 : 4;
}

// Plain rows on the matrix cores: whether they go there, parts of k that a tile's sixteen lines are dealt to, waves of a workgroup, LDS.
// Parts: as many as leave at most a workgroup per CU, four up to 1024 outputs, two up to 2048; bf16 from lengths on at which a tile's trip
// is long enough to halve (us, one / two / four parts: 4 rows of 768 x 768 3.5 / 4.0 / 3.7, 1024 x 1024 3.9 / 3.9 / 3.8, 2048 x 2048 4.7 / 4.9 / 5.2, 4096 x 2048
// 7.6 / 6.8 / 7.1, and four where the shares are two pairs that stay in registers, 5632 x 2048 10.1 / 8.7 / 8.0; 8 rows of 1024 x 1024 4.2 / 4.2, 2048 x
// 2048 5.6 / 5.2).  Beyond 4096 outputs a CU takes several tiles, and smaller ones even out their number: bf16 where that brings a wave's
// share down to two pairs, which stay in registers: up to 4 rows from 4096 of k to 8192 (4096 x 4608 12.7 / - / 10.5, x 12352 24.2 / 20.8 / 20.3; but 4096 x 4096 8.4 / 10.4 /
// 10.0), 8 rows beyond 2048 to 4096 (one / two: 2560 x 8192 13.0 / 10.8, x 12352 20.4 / 14.2, 3584 x 4608 13.3 / 11.0, x 22016 37.2 / 27.6, 4096 x 12352 24.8 / 20.4; 2048 x 12352 12.7 /
// 12.3 with shares that are two pairs already; longer ones are not, 4224 x 8192 17.0 / 24.1, 4608 x 12352 28.5 / 37.8, 6144 x 8192 22.2 / 29.9).
// f32 from 4096 on up to 5120 outputs, whose tiles of 16 leave the second round of workgroups nearly empty, if the waves' shares come out even, and
// wherever rows are 32 KiB apart (us, one part with sixteen waves / with eight / parts: 4 rows of 5632 x 5000 27.1 / 25.7 / 23.9, 8 of 8192 x 8192 50.7 / 62.2 /
// 50.4; but 4 of 5632 x 8192 30.5 / 29.3 / 36.8, 8704 x 8192 44.9 / 44.1 / 67.3, 11008 x 8192 60.2 / 62.3 / 71.2, 9216 x 4112 in uneven shares 39.3 / 39.0 / 40.1;
// 4096 x 9000 31.3 / 27.7 / 26.7 is the exception).
// Waves of one part, up to eight rows of bf16: eight rather than sixteen from 33 pairs on, two workgroups a CU, one of which asks while the other adds up (us,
// 16 / 8: 4 rows of 4224 x 4096 9.2 / 7.9, 11008 x 4112 28.0 / 25.5, one of 11008 x 3072 14.9 / 14.0, 8 of 2112 x 12352 21.2 / 15.7, 4608 x 9000 25.9 / 21.7; 10240 and
// 12288 - 24576 long 0.96 - 1.02 of the time; sixteen rows are not faster, 2048 x 1024 6.5 / 7.0).  Of 32 pairs, two for each of sixteen waves that stay in
// registers, as long as outputs are few (4 rows of 2048 x 6176 7.9 / 7.0, x 11264 0.93 of the time, x 12352 11.6 / 12.4; 8 of x 8192 0.90, x 9000 1.04, x 12352 1.12); of
// fewer as many as have two, or three where that comes out even, asked for at once (4 rows of 768 x 2304, two / three: 3.83 / 3.60; - x 10272 5.65 / 5.84, 1536 x 12352
// 8.5 / 10.7, 8 of 1536 x 5000 6.4 / 7.1).  Twelve of a multiple of 256 pairs, where eight begin a multiple of 4 KiB apart in rows a multiple of 32 KiB apart and share
// their memory channels (16 / 8 / 12: 4 rows of bf16 16384 x 3600 22.6 / 26.2 / 22.4, f32 8192 x 4096 27.4 / 30.0 / 24.0; 512 pairs x 2064 - 6176 0.85 - 1.02 of the time with eight, 768
// 0.92 - 0.98; 252 and 260 pairs 1.00 - 1.05).
// f32: eight (16 / 8: 4 rows of 768 x 3072 4.9 / 4.5, 1024 x 3600 6.1 / 5.3); four where there are several tiles a CU and rows are short of 4096 (16 / 8 / 4: 1024 x 4608 8.3 /
// 7.3 / 6.6, 2048 x 8192 15.0 / 13.8 / 13.7; but 4 rows of 8224 x 8192 48.1 / 46.2 / 60.1, 16 of 4096 x 8192 26.5 / 24.6 / 30.4) or 32 KiB apart (16 of 16384 x 4112 101 / 88 / 82).  Very many outputs of rows
// 96 to 512 long want as many waves as have two pairs in registers (time with four over that, mean of 2 - 16 rows: 128 x 50257 1.14, x 28747 1.11, 320 x 50257 1.12, 512 x
// 50257 1.04, but 20000 outputs of 96 - 512 0.98, 576 x 50257 0.92, 64 x 28747 0.93).
struct MfmaPlain { bool runs; uint32_t parts, waves; size_t lds; };
template <bool BF16>
static MfmaPlain gemv_mfma_plain(const Weight &w, uint64_t batch) {
    const uint32_t xbp = std::max(pad_batch(batch), 4u), most = 16 / xbp;  // (a part needs columns for all rows)
    auto fits = [&](uint32_t parts) { return parts <= most && w.k % (MfmaType<BF16>::KU * parts) == 0; };
    // f32: waves for that many parts; whether they ask for little in vain, two or three pairs at once
    auto f32_waves = [&](uint32_t parts) {
        const uint64_t pairs = std::min<uint64_t>(w.k / (MfmaType<false>::KU * parts), 1u << 20), four = std::max<uint64_t>(4, ceil_div(pairs, 4));
        uint64_t waves = gemv_mfma_waves(pairs);
        if (parts == 4) waves = pairs <= 12 ? std::max<uint64_t>(4, ceil_div(pairs, 2)) : std::min<uint64_t>(16, four);
        else if (parts == 2) waves = pairs >= 128 ? 16 : std::min<uint64_t>(8, four);
        else if (w.n > 4096) waves = pairs > 2 && pairs <= 16 && w.n > 20000 ? waves : pairs < 128 || pairs % 256 == 0 ? 4 : 8;
        else if (xbp < 16) waves = pairs % 256 == 0 ? 12 : std::min<uint64_t>(8, four);
        return (uint32_t)std::min<uint64_t>(waves, std::max<uint64_t>(1, pairs));
    };
    auto even = [&](uint32_t parts) {
        const uint64_t pairs = w.k / (MfmaType<false>::KU * parts), waves = f32_waves(parts), np = ceil_div(pairs, waves);
        return 4 * std::min(ceil_div(np, 2) * 2, ceil_div(np, 3) * 3) * waves <= 5 * pairs;
    };
    uint32_t parts = 1;
    if (BF16) {
        if (w.n <= 1024 && w.k >= 1024 && fits(4)) parts = 4;
        else if (w.n <= 2048 && w.k > 4096 && w.k <= 8192 && fits(4)) parts = 4;
        else if (w.n > 4096 && w.k >= 4096 && w.k <= 8192 && fits(4)) parts = 4;
        else if (((w.n <= 2048 && w.k >= (xbp == 8 || w.n <= 1024 ? 2048 : 4096)) || (w.n > 4096 && w.k > 2048 && w.k <= 4096 && xbp == 8)) && fits(2)) parts = 2;
    } else if (w.k >= 256) {
        auto wide = [&](uint32_t p) { return w.n > 4096 && w.k >= 4096 && (w.k % 8192 == 0 || (w.n <= 5120 && even(p))); };
        if (fits(4) && (w.n <= 1024 || wide(4))) parts = 4;
        else if (fits(2) && (w.n <= 2048 || wide(2))) parts = 2;
    }
    const uint64_t pairs = std::min<uint64_t>(w.k / (MfmaType<BF16>::KU * parts), 1u << 20);
    uint32_t waves = gemv_mfma_waves(pairs);
    if (BF16) {
        if (parts > 1) waves = pairs > 32 ? 8 : waves;
        else if (xbp == 4 && pairs % 3 == 0 && pairs >= 9 && pairs <= 24 && w.n <= 8192) waves = (uint32_t)std::max<uint64_t>(waves / 2, pairs / 3);
        else if (xbp <= 8 && (pairs > 32 || (pairs == 32 && w.n <= (xbp == 4 ? 12288 : 8192)))) waves = pairs % 256 == 0 ? 12 : 8;
    } else {
        waves = f32_waves(parts);
    }
    const uint32_t rows = parts > 1 ? 16 : xbp;
    const size_t lds = (size_t)waves * 16 * mfma_wave_lds<BF16>((rows + MfmaType<BF16>::XROWS - 1) / MfmaType<BF16>::XROWS);
    return {gemv_uses_mfma(w, batch, waves, false) && lds <= 160 * 1024, parts, waves, lds};
}

template <bool BF16>
static int launch_gemv_dense(const Weight &w, const float *x, uint64_t batch, const EpiArgs &e,
                             hipStream_t st, const NormFuse *nf) {
    const uint32_t bp = pad_batch(batch), b = (uint32_t)batch;
    if (nf && nf->streams) return launch_gemv_hyper<BF16>(w, batch, e, st, *nf);
    const bool post_norm = nf && nf->y;
    if (nf && !(post_norm ? gemv_can_fuse_post_norm(w, batch) : gemv_can_fuse_norm_dense(w, batch)))
        return fail(COEUS_INVALID_INPUT, "norm fusion needs the normalised activations to fit in LDS");
    if (post_norm && (!nf->h || !nf->scale || !nf->h_out || nf->h_out == nf->h || nf->kind != COEUS_NORM_RMSNORM))
        return fail(COEUS_INVALID_INPUT, "a norm behind the previous sublayer needs its output, the residual rows and "
                                         "a place for the new ones");
    if (nf && !post_norm && (!nf->h || !nf->scale))
        return fail(COEUS_INVALID_INPUT, "null pointer argument");
    // plain: 4 rows per workgroup; folded norm: 16, so that the block is normalised once per 16 rows
    const uint32_t waves = nf ? 16 : 4;
    const dim3 grid((unsigned)ceil_div(w.n, waves)), block(waves * 64);
    const int norm = !nf ? 0 : post_norm ? 3 : nf->whole ? 4 : nf->kind == COEUS_NORM_RMSNORM ? 2 : 1;
    const size_t lds = norm == 0 ? 0 : norm == 3 ? gemv_dense_post_lds(w.k, bp) : norm == 4 ? gemv_whole_norm_lds(w.k, bp) : gemv_dense_norm_lds(w.k, bp);
    if (norm == 4 && (!gemv_can_fuse_whole_norm(w, batch) || nf->kind != COEUS_NORM_LAYERNORM))
        return fail(COEUS_INVALID_INPUT, "a folded norm over all rows needs f32 weights, 2 to 16 rows and room in LDS");
    const uint64_t ldx = nf && nf->ld ? nf->ld : w.k;
    const PostNorm post = post_norm ? PostNorm{nf->y, nf->ls, nf->h_out} : PostNorm{nullptr, nullptr, nullptr};
    const float *xin = nf ? nf->h : x;
    const float *ns = nf ? nf->scale : nullptr, *nb = nf ? nf->bias : nullptr;
    const float eps = nf ? nf->eps : 0.f;
    // 16-byte loads
    const bool aligned = (((uintptr_t)xin | (uintptr_t)ns | (uintptr_t)nb | (uintptr_t)post.y | (uintptr_t)post.ls | (uintptr_t)post.h_out | (nf ? ldx * 4 : 0)) & 15) == 0;
    // (up to 1024 elements: a wave's registers hold the row, its scale and bias and four weight rows)
    if (bp == 1 && (norm == 1 || norm == 2) && aligned && w.k % 8 == 0 && w.k <= 1024 && w.n < (1ull << 31) - 64) {
#define COEUS_ROW(SV, RMSV) hipLaunchKernelGGL((gemv_row_kernel<BF16, RMSV, SV, kRowR>), dim3((unsigned)ceil_div(w.n, 4 * kRowR)), dim3(256), 0, st, w.data, xin, (uint32_t)w.k, ns, nb, eps, e)
        if (w.k <= 512) { if (norm == 1) COEUS_ROW(1, false); else COEUS_ROW(1, true); }
        else { if (norm == 1) COEUS_ROW(2, false); else COEUS_ROW(2, true); }
#undef COEUS_ROW
        COEUS_HIP(hipGetLastError());
        return COEUS_OK;
    }
    if (norm == 0 && aligned && gemv_takes_many(w, batch, epi_gated(e.act))) {
        const dim3 mgrid((unsigned)ceil_div(w.n, 8));
        if (w.k <= 1024) hipLaunchKernelGGL((gemv_many_kernel<BF16, 2>), mgrid, dim3(256), 0, st, w.data, xin, (uint32_t)w.k, e);
        else hipLaunchKernelGGL((gemv_many_kernel<BF16, 4>), mgrid, dim3(256), 0, st, w.data, xin, (uint32_t)w.k, e);
        COEUS_HIP(hipGetLastError());
        return COEUS_OK;
    }
    {
        // plain: workgroups enough to fill the compute units' 16 waves;
        // a folded norm: one workgroup of up to 16 waves per compute unit, which stages the rows once
        const uint32_t pairs = (uint32_t)std::min<uint64_t>(w.k / MfmaType<BF16>::KU, 1u << 20);
        const MfmaPlain plain = gemv_mfma_plain<BF16>(w, batch);
        const uint32_t mw = nf ? gemv_fold_waves(w) : plain.waves;
        const size_t mlds = nf ? gemv_mfma_norm_lds(w, bp, lds) : plain.lds;
        if (aligned && (nf ? gemv_folds_on_mfma(w, batch, lds) : plain.runs)) {
            const uint32_t parts = nf ? 1u : plain.parts, tiles = (uint32_t)ceil_div(w.n, 16 / parts), np = (pairs / parts + mw - 1) / mw;
            const dim3 mgrid(std::min(tiles, 256 * (16 / mw))), mblock(mw * 64);
#define COEUS_MFMA6(BPV, NV, PV, KV, TV, FV)                                                                                  \
    do {                                                                                                                      \
        static const bool once = [] { (void)hipFuncSetAttribute((const void *)gemv_mfma_kernel<BF16, BPV, NV, PV, KV, TV, FV>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); return true; }(); \
        (void)once;                                                                                                           \
        hipLaunchKernelGGL((gemv_mfma_kernel<BF16, BPV, NV, PV, KV, TV, FV>), mgrid, mblock, mlds, st, (const typename MfmaType<BF16>::W *)w.data, xin, (uint32_t)w.k, (uint32_t)w.n, b, mw, mgrid.x, e, ns, nb, eps, ldx, post); \
    } while (0)
#define COEUS_MFMA5(BPV, NV, PV, KV, TV) COEUS_MFMA6(BPV, NV, PV, KV, TV, false)
#define COEUS_MFMA4(BPV, NV, PV, KV) COEUS_MFMA5(BPV, NV, PV, KV, 1)
            // Pairs in flight: two or three, whichever asks for fewer in vain at the end of a wave's share.  Where that is the
            // same, three for 2 - 4 rows (us for two / three: 4 rows of bf16 5120 x 32000 67.0 / 65.5, 2 of 12288 x 8192 36.5 / 35.0), two
            // for one row (6144 x 512 7.2 / 7.4) and for 8 (6144 x 4096 13.0 / 13.5).  A norm in front fills the first trip, and
            // three pay from the second tile on (2 rows of bf16 3072 x 4096 12.7 / 13.3, x 12288 22.4 / 20.8).  Four in flight are
            // never faster (4 rows, us for 2 / 3 / 4: 3072 x 4096 7.1 / 6.4 / 7.1, 4096 x 4096 7.7 / 9.2 / 7.8, 10240 x 512 12.1 / 13.7 /
            // 14.0).
            const uint32_t by2 = (np + 1) / 2 * 2, by3 = (np + 2) / 3 * 3;
            const bool three = norm ? by3 < by2 && tiles > 256 : by3 < by2 || (by3 == by2 && batch > 1 && bp <= 4);
            // (sixteen lines of bf16 ask for sixteen rows of activations: three pairs of them spill)
#define COEUS_MFMAP(TV) do { if (np <= 2) COEUS_MFMA5(16 / TV, 0, 2, true, TV); else if (!BF16 && three) COEUS_MFMA5(16 / TV, 0, (BF16 ? 2 : 3), false, TV); else COEUS_MFMA5(16 / TV, 0, 2, false, TV); } while (0)
#define COEUS_MFMAL(BPV, NV, FV) do { if (BPV < 16 && three) COEUS_MFMA6(BPV < 16 ? BPV : 8, NV, 3, false, 1, FV); else COEUS_MFMA6(BPV, NV, 2, false, 1, FV); } while (0)
#define COEUS_MFMA3(BPV, NV) do { if (np <= 2) COEUS_MFMA4(BPV, NV, 2, true); else if (pairs > 4 * mw) COEUS_MFMAL(BPV, NV, (BF16 && NV == 0 && BPV < 16)); else COEUS_MFMAL(BPV, NV, false); } while (0)
#define COEUS_MFMAN(BPV, NV)                                                                               \
    do {                                                                                                   \
        if (BF16 && np == 1) COEUS_MFMA4(BPV, NV, (BF16 ? 1 : 2), true);                                    \
        else if constexpr (gemv_fold_share<BF16>(NV, BPV) > 2) COEUS_MFMA3(BPV, NV);                        \
        else if constexpr (gemv_fold_share<BF16>(NV, BPV) > (BF16 ? 1 : 0)) COEUS_MFMA4(BPV, NV, 2, true);  \
        else return fail(COEUS_INVALID_INPUT, "norm fusion needs the normalised activations to fit in LDS"); \
    } while (0)
#define COEUS_MFMA(BPV) do { if (norm == 4) { if constexpr (!BF16) COEUS_MFMAN(BPV, 4); } else if (norm == 1) COEUS_MFMAN(BPV, 1); else if (norm == 2) COEUS_MFMAN(BPV, 2); else COEUS_MFMAN(BPV, 3); } while (0)
            if (norm == 0 && parts == 4) COEUS_MFMAP(4);
            else if (norm == 0 && parts == 2) COEUS_MFMAP(2);
            else if (norm == 0 && bp <= 4) COEUS_MFMA3(4, 0);
            else if (norm == 0 && bp == 8) COEUS_MFMA3(8, 0);
            else if (norm == 0) COEUS_MFMA3(16, 0);
            else if (bp == 2) COEUS_MFMA(2);
            else if (bp == 4) COEUS_MFMA(4);
            else if (bp == 8) COEUS_MFMA(8);
            else COEUS_MFMA(16);
#undef COEUS_MFMA
#undef COEUS_MFMAN
#undef COEUS_MFMA3
#undef COEUS_MFMAL
#undef COEUS_MFMA4
#undef COEUS_MFMA5
#undef COEUS_MFMA6
#undef COEUS_MFMAP
            COEUS_HIP(hipGetLastError());
            return COEUS_OK;
        }
    }
    if (const uint32_t steps = norm == 0 && aligned ? gemv_one_row_steps(w, batch, epi_gated(e.act)) : 0) {
#define COEUS_ONE(DV) hipLaunchKernelGGL((gemv_dense_kernel<BF16, 1, 0, DV>), grid, block, 0, st, w.data, xin, w.k, b, e, ns, nb, eps, ldx, post)
        if (steps == 1) COEUS_ONE(1);
        else if (steps == 4) COEUS_ONE(4);
        else if constexpr (BF16) COEUS_ONE(6);
        else if (steps == 2) COEUS_ONE(2);
        else COEUS_ONE(3);
#undef COEUS_ONE
        COEUS_HIP(hipGetLastError());
        return COEUS_OK;
    }
    if (norm == 4) return fail(COEUS_INVALID_INPUT, "a folded norm over all rows needs its vectors on 16-byte boundaries");
#define COEUS_GEMVD2(BPV, NV) \
    hipLaunchKernelGGL((gemv_dense_kernel<BF16, BPV, NV>), grid, block, lds, st, w.data, xin, w.k, b, e, ns, nb, eps, ldx, post)
#define COEUS_GEMVD(BPV) \
    do { if (norm == 0) COEUS_GEMVD2(BPV, 0); else if (norm == 1) COEUS_GEMVD2(BPV, 1); else if (norm == 2) COEUS_GEMVD2(BPV, 2); else COEUS_GEMVD2(BPV, 3); } while (0)
    switch (bp) {
        case 1: COEUS_GEMVD(1); break;
        case 2: COEUS_GEMVD(2); break;
        case 4: COEUS_GEMVD(4); break;
        case 8: COEUS_GEMVD(8); break;
        default: COEUS_GEMVD(16); break;
    }
#undef COEUS_GEMVD
#undef COEUS_GEMVD2
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

coeus_matmul_plan gemv_plan(const Weight &w, uint64_t batch) {
    const uint32_t bp = pad_batch(batch);
    if (w.dtype >= COEUS_W_Q8_0) {
        if (!gemv_takes_rows(w, batch)) return {"gemv_quad_kernel", bp, 16, 0, 1, 1};
        uint32_t tpw, waves;
        gemv_rows_shape(w.dtype == COEUS_W_Q4_0, (uint32_t)(w.k_pad / 128), (uint32_t)(w.n_pad / 16), tpw, waves);
        return {"gemv_rows_kernel", bp, 16 * tpw, waves, 1, 1};
    }
    if (gemv_takes_many(w, batch)) return {"gemv_many_kernel", 1, 8, 4, 1, 1};
    const MfmaPlain mp = w.dtype == COEUS_W_BF16 ? gemv_mfma_plain<true>(w, batch) : gemv_mfma_plain<false>(w, batch);
    if (mp.runs) return {"gemv_mfma_kernel", bp, 16 / mp.parts, mp.waves, 1, 1};
    return {"gemv_dense_kernel", bp, 4, 4, 1, 1};
}

int launch_gemv(const Weight &w, const void *x, uint64_t batch, const Epilogue &ep, hipStream_t st,
                const NormFuse *nf) {
    if (batch == 0 || batch > 16)
        return fail(COEUS_INVALID_INPUT, "decode matmul batch %llu out of range [1, 16]",
                    (unsigned long long)batch);
    if (ep.act >= COEUS_EPI_CLAMP_GATE && w.dtype >= COEUS_W_Q8_0)
        return fail(COEUS_INVALID_INPUT, "epilogue %u takes f32 or bf16 weights", ep.act);
    if (epi_gated(ep.act) && (w.n & 1))
        return fail(COEUS_INVALID_INPUT, "gated epilogue needs an even number of weight rows");
    const EpiArgs e = make_epi(ep, w.n);
    if (e.g_out && (w.dtype < COEUS_W_Q8_0 || pad_batch(batch) > 4 || !e.g_scale || e.act == COEUS_EPI_SILU_GATE || e.kv_k))
        return fail(COEUS_INVALID_INPUT, "a pre-scaled copy of the output is written by the quantised decode matmul "
                                         "for batches of up to 4, without gate or cache append");
    switch (w.dtype) {
        case COEUS_W_F32: return launch_gemv_dense<false>(w, (const float *)x, batch, e, st, nf);
        case COEUS_W_BF16: return launch_gemv_dense<true>(w, (const float *)x, batch, e, st, nf);
        case COEUS_W_Q8_0: return launch_gemv_quant<false>(w, (const __half *)x, batch, e, st, nf);
        default: return launch_gemv_quant<true>(w, (const __half *)x, batch, e, st, nf);
    }
}

// ---------------------------------------------------------------- short prompts on quantised weights
// A prompt pass of up to 64 rows streams every weight once, like a decode step, so it should
// stream the Q4_0 / Q8_0 blocks and not their 3.5x larger f16 copies.  One workgroup takes 128
// weight rows (4 waves x 2 tiles of 16) over a share of at most GPW 128-wide k groups (blockIdx.y):
// all of its weights (2 x GPW chunks per wave) are requested first, the activation rows of the
// share (f16, from the previous kernel's 16-bit output) are staged in LDS once for all four
// waves, and after one barrier each wave unpacks its chunks to f16(q * d) (the same values as the
// f16 copies, so the results match the large-prompt path) and multiplies them with MT fragments
// of 16 activation rows (v_mfma_f32_16x16x32_f16; a fragment read from LDS feeds both tiles).
// No barrier and no request inside the multiply phase.  With more than one share the workgroups
// store bare partial products for gemm_split_reduce_kernel.
template <int GPW>
struct QsLayout {
    static constexpr int XLD = GPW * 128 + 8;  // LDS row stride in elements: + 8 keeps the 16-byte reads of 16 rows on distinct banks
};

template <bool Q4, int MT, int GPW>
__global__ __launch_bounds__(256) void gemm_qskinny_kernel(const uint16_t *__restrict__ a, uint64_t lda, uint32_t m,
                                                           const uint4 *__restrict__ qs,
                                                           const uint2 *__restrict__ ds, uint32_t tiles,
                                                           uint32_t ngroups, uint32_t splits, EpiArgs e) {
    constexpr int XLD = QsLayout<GPW>::XLD;
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];  // [MT * 16][XLD]
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t j = lane & 15, g = lane >> 4;
    const uint32_t split = blockIdx.y;
    const uint32_t gb = ngroups * split / splits, ge = ngroups * (split + 1) / splits;  // ge - gb <= GPW
    const uint32_t T0 = blockIdx.x * 8 + wave * 2;
    const uint64_t c0 = (uint64_t)min(T0, tiles - 1) * ngroups, c1 = (uint64_t)min(T0 + 1, tiles - 1) * ngroups;
    // Every load is unconditional (a load under a branch makes the compiler wait for all of them
    // before the first use): past the end of the share the last group is read again and multiplied
    // by a zero scale.
    ChunkRegs<Q4> rw[GPW][2];
#pragma unroll
    for (int d = 0; d < GPW; d++) {
        const uint32_t Gd = min(gb + d, ge - 1);
        load_chunk<Q4>(rw[d][0], qs, ds, c0 + Gd, lane);
        load_chunk<Q4>(rw[d][1], qs, ds, c1 + Gd, lane);
    }
    // activations: MT * 16 rows x GPW * 16 pieces of 16 bytes, 256 threads (rows past the end repeat
    // the last, groups past the share its last; m <= 64 rows: 32-bit offsets from the uniform base)
    constexpr int PPR = GPW * 16, NPT = MT * 16 * PPR / 256;  // pieces per row, pieces per thread
#pragma unroll
    for (int h = 0; h < NPT; h += 4) {
        uint4 v[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t p = tid + 256 * (h + q), row = p / PPR, pc = p % PPR;
            const uint32_t G = min(gb + pc / 16, ge - 1);
            v[q] = *(const uint4 *)(a + (min(row, m - 1) * (uint32_t)lda + G * 128 + (pc & 15) * 8));
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t p = tid + 256 * (h + q), row = p / PPR, pc = p % PPR;
            *(uint4 *)(xs + row * XLD + pc * 8) = v[q];
        }
    }
    float4_t acc[2][MT];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int u = 0; u < MT; u++) acc[t][u] = float4_t{0.f, 0.f, 0.f, 0.f};
    lds_barrier();
    const uint16_t *xb = xs + j * XLD + g * 8;
#pragma unroll
    for (int d = 0; d < GPW; d++) {
        const _Float16 live = gb + d < ge ? (_Float16)1.0f : (_Float16)0.0f;
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            half8_t wv[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const ChunkRegs<Q4> &r = rw[d][t];
                const uint32_t qw[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, Q4 ? 0u : r.q1.x, Q4 ? 0u : r.q1.y,
                                        Q4 ? 0u : r.q1.z, Q4 ? 0u : r.q1.w};
                union { uint2 u2; _Float16 h[4]; } sc;
                sc.u2 = r.s;
                const half8_t q = Q4 ? unpack_q4(qw[jj]) : unpack_q8(qw[2 * jj], qw[2 * jj + 1]);
                wv[t] = q * (sc.h[jj] * live);  // f16(q * d): one rounding, as in the dense f16 copy
            }
#pragma unroll
            for (int u = 0; u < MT; u++) {
                union { uint4 u4; half8_t h; } xv;
                xv.u4 = *(const uint4 *)(xb + u * 16 * XLD + d * 128 + jj * 32);
                acc[0][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv.h, wv[0], acc[0][u], 0, 0, 0);
                acc[1][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv.h, wv[1], acc[1][u], 0, 0, 0);
            }
        }
    }
    // lane (j, g) holds outputs (row 16 u + 4 g + i, column 16 T + j)
    if (splits > 1) {
        // Bare products into this share's plane (the usual case).  Through LDS, which is free now,
        // so that a row's 128 columns leave as 512 contiguous bytes instead of 16 floats per wave.
        constexpr uint32_t OLD = 132;  // floats per LDS row
        float *ts = (float *)xs;
        lds_barrier();  // (the last group's reads of xs are done)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int u = 0; u < MT; u++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    ts[(16 * u + 4 * g + i) * OLD + wave * 32 + t * 16 + j] = acc[t][u][i];
        lds_barrier();
        float *plane = e.out_f32 + (uint64_t)split * m * e.n;
        const uint64_t colbase = (uint64_t)blockIdx.x * 128;
        const uint32_t c4 = (tid & 31) * 4;
        for (uint32_t row = tid >> 5; row < MT * 16 && row < m; row += 8) {
            const float4 v = *(const float4 *)(ts + row * OLD + c4);
            float *dst = plane + (uint64_t)row * e.n + colbase + c4;
            if ((e.n & 3) == 0 && colbase + c4 + 3 < e.n) {
                *(float4 *)dst = v;
            } else {
                const float vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (colbase + c4 + q < e.n) dst[q] = vv[q];
            }
        }
        return;
    }
    const bool gated = e.act == COEUS_EPI_SILU_GATE;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint32_t T = T0 + t;
        const uint64_t col = (uint64_t)T * 16 + j;
#pragma unroll
        for (int u = 0; u < MT; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t row = 16 * u + 4 * g + i;
                // gated: weight rows (2c, 2c+1) = (gate_c, up_c) sit in neighbouring lanes
                const float other = lane_xor1(acc[t][u][i]);
                if (T >= tiles || row >= m || col >= e.n) continue;
                if (!gated) epi_store<false>(e, row, col, acc[t][u][i]);
                else if ((lane & 1) == 0) epi_store_gated(e, row, col >> 1, acc[t][u][i], other);
            }
    }
}

// k groups per workgroup: 4, or 2 when that takes the launch to at least 512 workgroups (narrow matrices).
static uint32_t qskinny_gpw(const Weight &w) {
    const uint32_t ngroups = (uint32_t)(w.k_pad / 128), tiles = (uint32_t)(w.n_pad / 16);
    const uint32_t wgs = (tiles + 7) / 8;
    return wgs * ((ngroups + 3) / 4) >= 512 ? 4 : 2;
}
uint32_t qskinny_splits(const Weight &w) {
    const uint32_t ngroups = (uint32_t)(w.k_pad / 128), gpw = qskinny_gpw(w);
    return (ngroups + gpw - 1) / gpw;
}

// Prompts of up to 16 rows: the decode step's kernels on the 16-bit rows that the prompt's producers leave.  The tiles of the longer prompts are mostly rows
// that are not there, and their launches on small matrices are shares of k with a second launch that sums them.
// Prompt passes, ms, those (gemm_narrow_kernel, gemm_qskinny_kernel) / these, of 2, 8 and 16 ids: 250M bf16 0.65 / 0.37, 0.66 / 0.42, 0.69 / 0.48; 250M Q8_0 0.64 /
// 0.38, 0.66 / 0.42, 0.65 / 0.41; 1B Q4_0 1.45 / 0.88, 1.54 / 1.03, 1.51 / 1.01; 7B Q4_0 2.52 / 1.68, 2.68 / 1.95, 2.82 / 2.03; matrix-memory layers 4096 wide
// 1.32 / 0.93, 1.32 / 0.98, 1.33 / 1.15.  The weights cross the memory interface once, so that beyond 16 rows these would read them twice.  Rules for waves and parts are the
// decode step's.  Errors to 64 bits of the same operands are smaller (bf16 11008 x 4096 9.1e-8, 1.6e-7 before, 768 x 2304 7.5e-8 and 8.4e-8; Q4_0 4096 x 4096 9.8e-8 and 1.3e-7).
bool gemm_uses_few(const Weight &w, uint64_t m) {
    if (m < 1 || m > 16 || w.dtype == COEUS_W_F32 || !w.few_rows) return false;
    if (w.dtype >= COEUS_W_Q8_0) return w.k == w.k_pad;
    return gemv_mfma_plain<true>(w, std::max<uint64_t>(m, 3)).runs;
}
coeus_matmul_plan gemm_few_plan(const Weight &w, uint64_t m) {
    const uint32_t bp = std::max(pad_batch(m), 4u);
    if (w.dtype == COEUS_W_BF16) {
        const MfmaPlain plain = gemv_mfma_plain<true>(w, std::max<uint64_t>(m, 3));
        return {"gemv_mfma_kernel", bp, 16 / plain.parts, plain.waves, 1, 1};
    }
    uint32_t tpw, waves;
    gemv_rows_shape(w.dtype == COEUS_W_Q4_0, (uint32_t)(w.k_pad / 128), (uint32_t)(w.n_pad / 16), tpw, waves);
    return {"gemv_rows_kernel", bp, 16 * tpw, waves, 1, 1};
}
int launch_gemm_few(const Weight &w, const uint16_t *a, uint64_t lda, uint64_t m, const EpiArgs &e, hipStream_t st) {
    if (w.dtype >= COEUS_W_Q8_0 && lda != gemm_ld(w.k)) return fail(COEUS_INVALID_INPUT, "matmul of few rows: rows %llu elements apart", (unsigned long long)lda);
    if (w.dtype == COEUS_W_Q8_0) return launch_gemv_rows_of<false, true>(w, a, m, e, st);
    if (w.dtype == COEUS_W_Q4_0) return launch_gemv_rows_of<true, true>(w, a, m, e, st);
    const MfmaPlain plain = gemv_mfma_plain<true>(w, std::max<uint64_t>(m, 3));
    const uint32_t bp = std::max(pad_batch(m), 4u), parts = plain.parts, mw = plain.waves, pairs = (uint32_t)(w.k / 64), np = (pairs / parts + mw - 1) / mw;
    const uint32_t tiles = (uint32_t)ceil_div(w.n, 16 / parts), rows = parts > 1 ? 16 : bp;
    const dim3 grid(std::min(tiles, 256 * (16 / mw))), block(mw * 64);
    const size_t lds = (size_t)mw * 16 * mfma_wave_lds<true, true>((int)ceil_div(rows, MfmaRows16::XROWS));
#define COEUS_FEW(BPV, KV, TV, FV)                                                                                             \
    do {                                                                                                                       \
        auto kern = gemv_mfma_kernel<true, BPV, 0, 2, KV, TV, FV, true>;                                                       \
        static const hipError_t room = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
        COEUS_HIP(room);                                                                                                       \
        hipLaunchKernelGGL(kern, grid, block, lds, st, (const uint16_t *)w.data, (const float *)a, (uint32_t)w.k, (uint32_t)w.n, (uint32_t)m, mw, grid.x, e, \
                           nullptr, nullptr, 0.f, lda, PostNorm{nullptr, nullptr, nullptr});                                   \
    } while (0)
#define COEUS_FEW2(BPV) do { if (np <= 2) COEUS_FEW(BPV, true, 1, false); else if (pairs > 4 * mw) COEUS_FEW(BPV, false, 1, true); else COEUS_FEW(BPV, false, 1, false); } while (0)
    if (parts == 4) { if (np <= 2) COEUS_FEW(4, true, 4, false); else COEUS_FEW(4, false, 4, false); }
    else if (parts == 2) { if (np <= 2) COEUS_FEW(8, true, 2, false); else COEUS_FEW(8, false, 2, false); }
    else if (bp == 4) COEUS_FEW2(4);
    else if (bp == 8) COEUS_FEW2(8);
    else COEUS_FEW2(16);
#undef COEUS_FEW2
#undef COEUS_FEW
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

// 17 to 64 rows (fewer: gemm_uses_few): with 128 (8 fragments of 16 rows per wave) the kernel needs 348 registers and
// is slower than the 256x256 kernel on the f16 copies.  Matrices of at least 4 M weights: below
// (the 250M shape) the 256x256 kernel split along k is as fast or faster.
bool gemm_uses_qskinny(const Weight &w, uint64_t m) {
    return w.dtype >= COEUS_W_Q8_0 && m > 16 && m <= 64 && w.k == w.k_pad && w.k >= 128 &&
           w.k * w.n >= 4000000ull;
}

uint64_t gemm_qskinny_scratch_bytes(const Weight &w, uint64_t m) {
    if (!gemm_uses_qskinny(w, m)) return 0;
    const uint32_t s = qskinny_splits(w);
    return s > 1 ? (uint64_t)s * m * w.n * 4 : 0;
}

// `plain` is the epilogue of a k-split launch (bare products into planes of `partials`); the caller
// runs the reduce kernel with the real epilogue afterwards.  Returns the number of shares used.
int launch_gemm_qskinny(const Weight &w, const uint16_t *a, uint64_t lda, uint64_t m, const EpiArgs &e,
                        float *partials, uint64_t partials_bytes, uint32_t *splits_out, hipStream_t st) {
    const uint32_t ngroups = (uint32_t)(w.k_pad / 128), tiles = (uint32_t)(w.n_pad / 16);
    const uint32_t splits = qskinny_splits(w);
    if (splits > 1 && (!partials || partials_bytes < (uint64_t)splits * m * w.n * 4))
        return fail(COEUS_INVALID_INPUT, "short-prompt matmul needs %llu bytes for its partial products",
                    (unsigned long long)((uint64_t)splits * m * w.n * 4));
    *splits_out = splits;
    EpiArgs ke = e;
    if (splits > 1) {
        Epilogue pe;
        pe.out_f32 = partials;
        ke = make_epi(pe, w.n);
    }
    const dim3 grid((tiles + 7) / 8, splits);
    const uint4 *qs = (const uint4 *)w.data;
    const uint2 *ds = (const uint2 *)w.scales;
    const bool q4 = w.dtype == COEUS_W_Q4_0;
#define COEUS_QS(Q4V, MTV, GPWV)                                                                        \
    do {                                                                                                \
        constexpr int lds_bytes = MTV * 16 * QsLayout<GPWV>::XLD * 2;                                    \
        static const bool once = [] {                                                                   \
            (void)hipFuncSetAttribute((const void *)gemm_qskinny_kernel<Q4V, MTV, GPWV>,                \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);            \
            return true;                                                                                \
        }();                                                                                            \
        (void)once;                                                                                     \
        hipLaunchKernelGGL((gemm_qskinny_kernel<Q4V, MTV, GPWV>), grid, dim3(256), (size_t)lds_bytes, st, a, lda, \
                           (uint32_t)m, qs, ds, tiles, ngroups, splits, ke);                            \
    } while (0)
#define COEUS_QS3(MTV, GPWV) do { if (q4) COEUS_QS(true, MTV, GPWV); else COEUS_QS(false, MTV, GPWV); } while (0)
#define COEUS_QS2(MTV) do { if (gpw == 4) COEUS_QS3(MTV, 4); else COEUS_QS3(MTV, 2); } while (0)
    const uint32_t gpw = qskinny_gpw(w);
    if (m <= 32) COEUS_QS2(2);
    else COEUS_QS2(4);
#undef COEUS_QS3
#undef COEUS_QS2
#undef COEUS_QS
    COEUS_HIP(hipGetLastError());
    return COEUS_OK;
}

}  // namespace coeus
