// Attention and the KV cache: RoPE + KV store, decode attention (one workgroup per head; cells split over several workgroups and
// merged), attention of prompt chunks on the matrix cores, K-shift and cache compaction.
#include "attn_decode.hpp"

namespace {

// ---------------------------------------------------------------------------------------------------
// K-shift (llm_build_k_shift, llama.cpp:4332-4381): cached K rows whose position changed by delta[cell] are rotated in place
// by that many positions, the RoPE of fp16 data (ggml_compute_forward_rope_f16, ggml.c:11327-11478): fp16 -> fp32, angle
// delta * theta_i with theta advanced by repeated fp32 multiplication, back to fp16.  Cache layout [row][n_ctx][hd] with
// row = (layer, kv head).  grid = (cells, rows), hd/2 threads; cells with delta 0 are left alone (the reference rotates them
// by angle 0, which returns the same bits).
// ---------------------------------------------------------------------------------------------------
__global__ void k_shift_kernel(__half * __restrict__ k_cache, int n_ctx, int hd, int mode, float theta_scale, float freq_scale,
                               const int32_t * __restrict__ delta) {
    const int cell = blockIdx.x, i = threadIdx.x;
    const int dl = delta[cell];
    if (dl == 0) return;
    __half * row = k_cache + ((size_t)blockIdx.y * n_ctx + cell) * hd;
    const float theta = rope_angle((float)dl, i, mode, theta_scale, freq_scale);
    const float c = cosf(theta), sn = sinf(theta);
    const int i0 = (mode & 2) ? i : 2 * i;
    const int i1 = (mode & 2) ? i + hd / 2 : 2 * i + 1;
    const float x0 = __half2float(row[i0]), x1 = __half2float(row[i1]);
    row[i0] = __float2half_rn(__fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, sn)));
    row[i1] = __float2half_rn(__fadd_rn(__fmul_rn(x0, sn), __fmul_rn(x1, c)));
}

// the same on the reference's own layout, K cells [layer][cell][kv head][hd]: grid = (cells, layers * kv heads)
__global__ void k_shift_cells_kernel(__half * __restrict__ k_cache, int n_cells, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                                     const int32_t * __restrict__ delta) {
    const int cell = blockIdx.x, i = threadIdx.x;
    const int dl = delta[cell];
    if (dl == 0) return;
    const int layer = blockIdx.y / n_head_kv, kvh = blockIdx.y % n_head_kv;
    __half * row = k_cache + (((size_t)layer * n_cells + cell) * n_head_kv + kvh) * hd;
    const float theta = rope_angle((float)dl, i, mode, theta_scale, freq_scale);
    const float c = cosf(theta), sn = sinf(theta);
    const int i0 = (mode & 2) ? i : 2 * i;
    const int i1 = (mode & 2) ? i + hd / 2 : 2 * i + 1;
    const float x0 = __half2float(row[i0]), x1 = __half2float(row[i1]);
    row[i0] = __float2half_rn(__fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, sn)));
    row[i1] = __float2half_rn(__fadd_rn(__fmul_rn(x0, sn), __fmul_rn(x1, c)));
}

// Cell compaction of one cache (K or V) after cells were removed: new cell j takes old cell map[j] (map ascending, so the cells
// keep their order).  Two launches through a staging buffer [rows][n_new][hd] because source and destination ranges overlap.
// grid = (n_new, rows), hd/8 threads (16 bytes each).
__global__ void kv_gather_kernel(const __half * __restrict__ cache, __half * __restrict__ stage, const int32_t * __restrict__ map, int n_new, int n_ctx, int hd) {
    const pi_u32x4 * src = reinterpret_cast<const pi_u32x4 *>(cache + ((size_t)blockIdx.y * n_ctx + map[blockIdx.x]) * hd);
    pi_u32x4 * dst = reinterpret_cast<pi_u32x4 *>(stage + ((size_t)blockIdx.y * n_new + blockIdx.x) * hd);
    dst[threadIdx.x] = src[threadIdx.x];
}
__global__ void kv_place_kernel(__half * __restrict__ cache, const __half * __restrict__ stage, int n_new, int n_ctx, int hd) {
    const pi_u32x4 * src = reinterpret_cast<const pi_u32x4 *>(stage + ((size_t)blockIdx.y * n_new + blockIdx.x) * hd);
    pi_u32x4 * dst = reinterpret_cast<pi_u32x4 *>(cache + ((size_t)blockIdx.y * n_ctx + blockIdx.x) * hd);
    dst[threadIdx.x] = src[threadIdx.x];
}

// ---------------------------------------------------------------------------------------------------
// RoPE + KV store for one token (ggml.c:11163-11325; theta advanced by repeated fp32 multiplication as
// the CPU path does, so the angle is bit-identical and only cosf/sinf may differ in the last place).
// grid = n_head + 2*n_head_kv blocks of hd/2 threads.
// ---------------------------------------------------------------------------------------------------
__global__ void rope_kv_store_kernel(const float * __restrict__ qkv, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                                     const int32_t * __restrict__ pos_p, int n_ctx, float * __restrict__ q_rot,
                                     __half * __restrict__ k_cache, __half * __restrict__ v_cache, int qkv_stride, int q_stride) {
    // blockIdx.y = token of a prompt chunk (same sequence, its own position); 0 for single-token decoding
    qkv += (size_t)blockIdx.y * qkv_stride;
    q_rot += (size_t)blockIdx.y * q_stride;
    pos_p += blockIdx.y;
    const int h = blockIdx.x, i = threadIdx.x;           // i = pair index
    const int pos = *pos_p;
    if (h < n_head + n_head_kv) {
        const float * src = qkv + (size_t)h * hd;
        const float theta = rope_angle((float)pos, i, mode, theta_scale, freq_scale);
        const float c = cosf(theta), s = sinf(theta);
        const int i0 = (mode & 2) ? i : 2 * i;
        const int i1 = (mode & 2) ? i + hd / 2 : 2 * i + 1;
        const float x0 = src[i0], x1 = src[i1];
        const float y0 = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, s));
        const float y1 = __fadd_rn(__fmul_rn(x0, s), __fmul_rn(x1, c));
        if (h < n_head) {
            q_rot[(size_t)h * hd + i0] = y0;
            q_rot[(size_t)h * hd + i1] = y1;
        } else {
            __half * dst = k_cache + ((size_t)(h - n_head) * n_ctx + pos) * hd;
            dst[i0] = __float2half_rn(y0);
            dst[i1] = __float2half_rn(y1);
        }
    } else {
        const int hv = h - n_head - n_head_kv;
        const float * src = qkv + (size_t)(n_head + n_head_kv + hv) * hd;
        __half * dst = v_cache + ((size_t)hv * n_ctx + pos) * hd;
        dst[2 * i]     = __float2half_rn(src[2 * i]);
        dst[2 * i + 1] = __float2half_rn(src[2 * i + 1]);
    }
}

// ---------------------------------------------------------------------------------------------------
// Decode attention: one block per query head over cells [0, pos].
// ---------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void attn_decode_kernel(const float * __restrict__ q_rot, const __half * __restrict__ k_cache,
                                                             const __half * __restrict__ v_cache, int n_head, int n_head_kv, int hd,
                                                             int n_ctx, const int32_t * __restrict__ pos_p, float * __restrict__ out,
                                                             int q_stride, int out_stride, __half * __restrict__ out16) {
    // blockIdx.y = token of a prompt chunk: it sees the cache cells up to its own position (causal mask)
    q_rot += (size_t)blockIdx.y * q_stride;
    out += (size_t)blockIdx.y * out_stride;
    if (out16) out16 += (size_t)blockIdx.y * out_stride;
    pos_p += blockIdx.y;
    extern __shared__ __align__(16) unsigned char smem[];
    float * s    = reinterpret_cast<float *>(smem);               // [n_kv] scores, then probabilities
    float * part = s + n_ctx;                                     // [groups][hd] partial outputs
    __shared__ double red[16];
    __shared__ float redf[16];
    const int h = blockIdx.x, kvh = h / (n_head / n_head_kv);
    const int n_kv = *pos_p + 1;
    const int lpp = hd / 8;                                       // lanes per position (16 B each)
    const int tid = threadIdx.x;
    const int sub = tid % lpp, grp = tid / lpp, ngrp = blockDim.x / lpp;
    const float scale = pi_inv_sqrt((float)hd);

    // q chunk of this lane, rounded to fp16 as the CPU dot does
    float qf[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) qf[i] = pi_round_f16(q_rot[(size_t)h * hd + sub * 8 + i]);

    const __half * kb = k_cache + (size_t)kvh * n_ctx * hd;
    for (int c0 = 0; c0 < n_kv; c0 += ngrp) {
        const int c = c0 + grp;
        float d = 0.0f;
        if (c < n_kv) d = pi_dot8(pi_ld16(kb + (size_t)c * hd + sub * 8), qf, 0.0f);
        for (int o = lpp / 2; o > 0; o >>= 1) d += __shfl_xor(d, o, PI_WAVE);
        if (c < n_kv && sub == 0) s[c] = __fmul_rn(d, scale);
    }
    __syncthreads();

    float mx = -INFINITY;
    for (int c = tid; c < n_kv; c += blockDim.x) mx = fmaxf(mx, s[c]);
    mx = block_max_f32(mx, redf);
    double sum = 0.0;
    for (int c = tid; c < n_kv; c += blockDim.x) {
        // exp through fp16 in and out: the CPU path's lookup table holds fp16(expf(fp32(fp16(x - max))))
        const float e = pi_round_f16(expf(pi_round_f16(__fsub_rn(s[c], mx))));
        s[c] = e;
        sum += (double)e;
    }
    sum = block_sum_f64(sum, red);                                // includes the barriers that publish s[]
    const float inv = (float)(1.0 / sum);

    const __half * vb = v_cache + (size_t)kvh * n_ctx * hd;
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    for (int c = grp; c < n_kv; c += ngrp) {
        const float p = pi_round_f16(__fmul_rn(s[c], inv));       // probabilities are rounded to fp16 before the V product
        float vf[8];
        pi_unpack8(pi_ld16(vb + (size_t)c * hd + sub * 8), vf);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = fmaf(vf[i], p, acc[i]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) part[grp * hd + sub * 8 + i] = acc[i];
    __syncthreads();
    for (int e = tid; e < hd; e += blockDim.x) {
        float v = part[e];
        for (int g = 1; g < ngrp; ++g) v += part[g * hd + e];
        out[(size_t)h * hd + e] = v;
        if (out16) out16[(size_t)h * hd + e] = __float2half_rn(v);
    }
}

// cos/sin of every (position, pair) the way the CPU path forms them: theta advanced by repeated fp32
// multiplication (ggml.c:11269-11319), so the angle is bit-identical and only cosf/sinf can differ in the
// last place.  table[p][i] = (cos, sin) for pair i of position p.
// Workgroups from n_head on (a single sequence only) request weights of later launches and take no part (load_ahead).
template <int BLOCK, int LPP>
__global__ __launch_bounds__(BLOCK, 8) void attn_fused_kernel(const float * __restrict__ qkv, const float2 * __restrict__ rope_table,
                                                            __half * __restrict__ k_cache, __half * __restrict__ v_cache,
                                                            int n_head, int n_head_kv, int hd, int mode, int n_ctx,
                                                            const int32_t * __restrict__ pos_p, float * __restrict__ out,
                                                            int qkv_stride, size_t cache_seq_stride, int out_stride, __half * __restrict__ out16, int out16_ol,
                                                            int8_t * __restrict__ q8_q, float * __restrict__ q8_d, int * __restrict__ q8_s, Ahead ahead) {
    if ((int)blockIdx.x >= n_head) { load_ahead(ahead, (int)blockIdx.x - n_head); return; }
    attn_fused_head<BLOCK, LPP>(qkv, rope_table, k_cache, v_cache, n_head, n_head_kv, hd, mode, n_ctx, pos_p, out, qkv_stride, cache_seq_stride, out_stride, out16, out16_ol, q8_q, q8_d, q8_s,
                                blockIdx.x, blockIdx.y);
}
// Attention and output projection of a small model's token: a head's workgroup multiplies what it attended with its columns of wo, whose rows travel under the attention, and leaves
// a vector of the model's width; ffn_small_f16_kernel adds the heads'.  Bound by latency like the attention alone: 7.3 us at 20
// cells where that takes 7.0 and the projection 3.4 behind it (the FFN then takes 9.1 instead of 8.2).  8 tokens of three layers of 512 x 4096, 8 heads: 790 -> 705 us at 20 cells, 830 -> 750
// at 300.
constexpr int kOutPre = 4;              // rows of wo a group of lanes requests ahead
template <int LPP>
__global__ __launch_bounds__(kAttnBlock, 4) void attn_out_small_kernel(const float * __restrict__ qkv, const float2 * __restrict__ rope_table, __half * __restrict__ k_cache, __half * __restrict__ v_cache,
                                                                       int n_head, int n_head_kv, int hd, int mode, int n_ctx, const int32_t * __restrict__ pos_p, const __half * __restrict__ wo, int d,
                                                                       float * __restrict__ parts) {
    __shared__ __align__(16) __half att[LPP * 8];
    const int h = blockIdx.x, sub = threadIdx.x % LPP, grp = threadIdx.x / LPP;
    constexpr int kGroups = kAttnBlock / LPP;
    const __half * w = wo + (size_t)h * hd + sub * 8;
    auto row = [&](int r) { return pi_ld16(w + (size_t)min(r, d - 1) * ((size_t)n_head * hd)); };
    pi_u32x4 ahead[kOutPre];
#pragma unroll
    for (int k = 0; k < kOutPre; ++k) ahead[k] = row(grp + k * kGroups);
    attn_fused_head<kAttnBlock, LPP>(qkv, rope_table, k_cache, v_cache, n_head, n_head_kv, hd, mode, n_ctx, pos_p, nullptr, 0, 0, 0, nullptr, 0, nullptr, nullptr, nullptr, h, 0, att);
    __syncthreads();
    const pi_u32x4 a = *reinterpret_cast<const pi_u32x4 *>(att + sub * 8);
    float * out = parts + (size_t)h * d;
    for (int r0 = grp; r0 < d; r0 += kOutPre * kGroups) {
        if (r0 != grp)
#pragma unroll
            for (int k = 0; k < kOutPre; ++k) ahead[k] = row(r0 + k * kGroups);
#pragma unroll
        for (int k = 0; k < kOutPre; ++k) {
            const float v = pi_group_sum<LPP>(pi_dot8h(ahead[k], a, 0.0f), LPP);
            if (sub == 0 && r0 + k * kGroups < d) out[r0 + k * kGroups] = v;
        }
    }
}
template <bool FROM_CACHE, int LPP>
__global__ __launch_bounds__(kAttnPartBlock, 4) void attn_part_kernel(const float * __restrict__ qkv, const float2 * __restrict__ rope_table,
                                                                   __half * __restrict__ k_cache, __half * __restrict__ v_cache,
                                                                   int n_head, int n_head_kv, int hd, int mode, int n_ctx, int s_cap,
                                                                   const int32_t * __restrict__ pos_p, float * __restrict__ part_acc, float * __restrict__ part_ml,
                                                                   int qkv_stride, size_t cache_seq_stride) {
    attn_part_head<FROM_CACHE, LPP>(qkv, rope_table, k_cache, v_cache, n_head, n_head_kv, hd, mode, n_ctx, s_cap, pos_p, part_acc, part_ml, qkv_stride, cache_seq_stride,
                                    blockIdx.x, blockIdx.y, gridDim.y, blockIdx.z);
}

// one workgroup of hd threads per head
__global__ void attn_merge_kernel(const float * __restrict__ part_acc, const float * __restrict__ part_ml, int n_parts, int hd,
                                  float * __restrict__ out, int out_stride, __half * __restrict__ out16) {
    const size_t h = blockIdx.x, t = blockIdx.y;
    const float v = attn_merge_value<false>(part_acc, part_ml, n_parts, hd, (t * gridDim.x + h) * n_parts, threadIdx.x);
    out[t * out_stride + h * hd + threadIdx.x] = v;
    if (out16) out16[t * out_stride + h * hd + threadIdx.x] = __float2half_rn(v);
}

// ---------------------------------------------------------------------------------------------------
// Attention of a prompt chunk on the matrix cores: a workgroup owns 16 consecutive tokens of one query head and the four waves
// split the cache cells.  Three phases, with the rounding points of attn_decode_kernel (and so of the CPU path):
//   1. scores: S[cell][token] = K[cell] . fp16(q[token]) by 16x16x32 MFMAs (a K row is read in operand layout straight from
//      the cache, q stays in registers), times 1/sqrt(hd), into LDS as s[token][cell];
//   2. softmax per token over the cells it may see (cell <= its position): maximum, fp16(exp(fp16(s - max))), the sum in double,
//      p = fp16(e / sum); cells beyond the token's position become exact zeros;
//   3. out[token][:] = sum over cells of p * V[cell][:]: the V cache keeps a cell's head contiguous, the MFMA wants eight cells of
//      one column per lane, so a wave reads eight cells of a column pair (4 bytes per lane, a whole row per instruction), packs
//      them with two byte permutes per pair of cells and drops two 16-byte columns into its private LDS tile (32 cells a tile),
//      from where the operand comes back with one 16-byte read.  No workgroup barrier inside the loops: the tile belongs to one
//      wave and the LDS operations of a wave complete in order.  The waves' partial outputs meet in LDS in wave order.
// q8: what the output matrix of a Q4_0 model multiplies with instead of the output, its values rounded through blocks of eight bits, by rows (1) or in
// the operand layout (2); a launch of 5.2 us for 130 tokens of 4096 columns otherwise.
// HD = 128 or 64.  LDS: 16 x (cells rounded up to 32, + 4) floats of scores + 4 x HD x 80 bytes of V tiles.
// ---------------------------------------------------------------------------------------------------
constexpr int kAcVtStride = 40;                // halves per row of the transposed V tile: 32 cells + 8 of padding (conflict-free both ways)
template <int HD>
__global__ __launch_bounds__(kBlock) void attn_chunk_mfma_kernel(const float * __restrict__ q_rot, const __half * __restrict__ k_cache,
                                                                 const __half * __restrict__ v_cache, int n_head, int n_head_kv, int n_ctx,
                                                                 const int32_t * __restrict__ pos_p, int T, float * __restrict__ out,
                                                                 int q_stride, int out_stride, __half * __restrict__ out16, int s_stride, int q8) {
    static_assert(HD == 128 || HD == 64, "head size");
    extern __shared__ __align__(16) unsigned char smem[];
    float * s = reinterpret_cast<float *>(smem);                                       // [16][s_stride]
    unsigned char * vt_all = smem + sizeof(float) * 16 * (size_t)s_stride;             // [4 waves][HD][kAcVtStride] halves
    const int h = blockIdx.x, kvh = h / (n_head / n_head_kv);
    const int t0 = blockIdx.y * 16;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    // cells the furthest-reaching token of the tile sees
    int n_kv = pos_p[min(t0 + i, T - 1)] + 1;
    for (int o = 8; o > 0; o >>= 1) n_kv = max(n_kv, __shfl_xor(n_kv, o, PI_WAVE));
    n_kv = min(n_kv, s_stride - 4);                // the launcher sized the scores for the cells its caller announced
    const int n_t16 = (n_kv + 15) / 16, n_t32 = (n_kv + 31) / 32;

    // ---- 1. scores --------------------------------------------------------------------------------------------------------
    {
        const float * qp = q_rot + (size_t)min(t0 + i, T - 1) * q_stride + (size_t)h * HD + 8 * g;
        pi_h8 qf[HD / 32];
#pragma unroll
        for (int ks = 0; ks < HD / 32; ++ks) {
            const float4 a = *reinterpret_cast<const float4 *>(qp + ks * 32), b = *reinterpret_cast<const float4 *>(qp + ks * 32 + 4);
            qf[ks] = pi_h8{(_Float16)a.x, (_Float16)a.y, (_Float16)a.z, (_Float16)a.w, (_Float16)b.x, (_Float16)b.y, (_Float16)b.z, (_Float16)b.w};
        }
        const float scale = pi_inv_sqrt((float)HD);
        const __half * kb = k_cache + (size_t)kvh * n_ctx * HD + 8 * g;
        // six tiles of K rows are in flight per wave: the loads come from L2 and a wave has little else to hide their latency behind
        constexpr int D1 = 6;
        pi_u32x4 a[D1][HD / 32];
        // (requests past the last tile re-read the last cell: unconditional loads keep the count of outstanding ones static, which
        // is what lets the compiler wait for the oldest tile only)
        auto issue = [&](pi_u32x4 * dst, int kt) {
            const int c = min(kt * 16 + i, n_kv - 1);
#pragma unroll
            for (int ks = 0; ks < HD / 32; ++ks) dst[ks] = pi_ld16(kb + (size_t)c * HD + ks * 32);
        };
#pragma unroll
        for (int u = 0; u < D1; ++u) issue(a[u], wave + u * kWavesPerBlock);
        for (int kt0 = wave; kt0 < n_t16; kt0 += D1 * kWavesPerBlock) {
#pragma unroll
            for (int u = 0; u < D1; ++u) {
                const int kt = kt0 + u * kWavesPerBlock;
                if (kt < n_t16) {
                    pi_f4 acc = pi_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int ks = 0; ks < HD / 32; ++ks) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(pi_h8, a[u][ks]), qf[ks], acc, 0, 0, 0);
                    // acc[r] = S[cell kt*16 + 4g + r][token i]
                    *reinterpret_cast<float4 *>(s + (size_t)i * s_stride + kt * 16 + 4 * g) =
                        float4{__fmul_rn(acc[0], scale), __fmul_rn(acc[1], scale), __fmul_rn(acc[2], scale), __fmul_rn(acc[3], scale)};
                }
                issue(a[u], kt + D1 * kWavesPerBlock);
            }
        }
    }
    __syncthreads();

    // ---- 2. softmax: 16 lanes per token, four cells per lane and step ------------------------------------------------------------
    {
        const int q = threadIdx.x >> 4, j = threadIdx.x & 15;
        const int nq = min(pos_p[min(t0 + q, T - 1)] + 1, n_kv);
        float * sq = s + (size_t)q * s_stride;
        float mx = -INFINITY;
        for (int c = 4 * j; c < nq; c += 64) {
            const float4 v = *reinterpret_cast<const float4 *>(sq + c);
            mx = fmaxf(mx, v.x);
            if (c + 1 < nq) mx = fmaxf(mx, v.y);
            if (c + 2 < nq) mx = fmaxf(mx, v.z);
            if (c + 3 < nq) mx = fmaxf(mx, v.w);
        }
        for (int o = 8; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, PI_WAVE));
        double sum = 0.0;
        for (int c = 4 * j; c < nq; c += 64) {
            float4 v = *reinterpret_cast<const float4 *>(sq + c);
            // exp through fp16 in and out, as the CPU path's lookup table does; cells past the token's own position count as zero
            v.x = pi_round_f16(expf(pi_round_f16(__fsub_rn(v.x, mx))));
            v.y = c + 1 < nq ? pi_round_f16(expf(pi_round_f16(__fsub_rn(v.y, mx)))) : 0.0f;
            v.z = c + 2 < nq ? pi_round_f16(expf(pi_round_f16(__fsub_rn(v.z, mx)))) : 0.0f;
            v.w = c + 3 < nq ? pi_round_f16(expf(pi_round_f16(__fsub_rn(v.w, mx)))) : 0.0f;
            *reinterpret_cast<float4 *>(sq + c) = v;
            sum += (double)v.x; sum += (double)v.y; sum += (double)v.z; sum += (double)v.w;
        }
        for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, PI_WAVE);
        const float inv = (float)(1.0 / sum);
        for (int c = 4 * j; c < n_t32 * 32; c += 64) {
            float4 v = float4{0.0f, 0.0f, 0.0f, 0.0f};
            if (c < nq) {
                v = *reinterpret_cast<const float4 *>(sq + c);
                v.x = pi_round_f16(__fmul_rn(v.x, inv)); v.y = pi_round_f16(__fmul_rn(v.y, inv));
                v.z = pi_round_f16(__fmul_rn(v.z, inv)); v.w = pi_round_f16(__fmul_rn(v.w, inv));       // zeros past nq stay zeros
            }
            *reinterpret_cast<float4 *>(sq + c) = v;
        }
    }
    __syncthreads();

    // ---- 3. p . V -------------------------------------------------------------------------------------------------------------
    pi_f4 acc[HD / 16];
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) acc[dt] = pi_f4{0.0f, 0.0f, 0.0f, 0.0f};
    unsigned char * myvt = vt_all + (size_t)wave * HD * kAcVtStride * 2;
    {
        constexpr int LPR = HD / 2;                 // lanes per V row, 4 bytes (a column pair) each
        constexpr int GPI = PI_WAVE / LPR;          // groups of eight cells per load instruction
        const int dp = lane % LPR, sub = lane / LPR;
        const __half * vb = v_cache + (size_t)kvh * n_ctx * HD + 2 * dp;
        // the cells of the next three tiles are on their way while a tile is packed and multiplied; cells past the end may hold
        // anything and enter as zeros
        constexpr int D3 = 3;
        unsigned vq[D3][4 / GPI][8];
        auto issue = [&](unsigned (*dst)[8], int kt) {
#pragma unroll
            for (int rnd = 0; rnd < 4 / GPI; ++rnd)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int c = kt * 32 + (rnd * GPI + sub) * 8 + k;
                    dst[rnd][k] = *reinterpret_cast<const unsigned *>(vb + (size_t)min(c, n_kv - 1) * HD);
                }
        };
#pragma unroll
        for (int u = 0; u < D3; ++u) issue(vq[u], wave + u * kWavesPerBlock);
        for (int kt0 = wave; kt0 < n_t32; kt0 += D3 * kWavesPerBlock) {
#pragma unroll
            for (int u = 0; u < D3; ++u) {
                const int kt = kt0 + u * kWavesPerBlock;
                if (kt < n_t32) {
                    const int c0 = kt * 32;
#pragma unroll
                    for (int rnd = 0; rnd < 4 / GPI; ++rnd) {
                        const int grp8 = rnd * GPI + sub;   // which eight cells of the tile
                        unsigned v[8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) v[k] = c0 + grp8 * 8 + k < n_kv ? vq[u][rnd][k] : 0u;
                        pi_u32x4 lo, hi;
                        lo.x = __builtin_amdgcn_perm(v[1], v[0], 0x05040100u); hi.x = __builtin_amdgcn_perm(v[1], v[0], 0x07060302u);
                        lo.y = __builtin_amdgcn_perm(v[3], v[2], 0x05040100u); hi.y = __builtin_amdgcn_perm(v[3], v[2], 0x07060302u);
                        lo.z = __builtin_amdgcn_perm(v[5], v[4], 0x05040100u); hi.z = __builtin_amdgcn_perm(v[5], v[4], 0x07060302u);
                        lo.w = __builtin_amdgcn_perm(v[7], v[6], 0x05040100u); hi.w = __builtin_amdgcn_perm(v[7], v[6], 0x07060302u);
                        *reinterpret_cast<pi_u32x4 *>(myvt + ((size_t)(2 * dp) * kAcVtStride + grp8 * 8) * 2) = lo;
                        *reinterpret_cast<pi_u32x4 *>(myvt + ((size_t)(2 * dp + 1) * kAcVtStride + grp8 * 8) * 2) = hi;
                    }
                    const float * pp = s + (size_t)i * s_stride + c0 + 8 * g;
                    const float4 p0 = *reinterpret_cast<const float4 *>(pp), p1 = *reinterpret_cast<const float4 *>(pp + 4);
                    const pi_h8 pa = pi_h8{(_Float16)p0.x, (_Float16)p0.y, (_Float16)p0.z, (_Float16)p0.w, (_Float16)p1.x, (_Float16)p1.y, (_Float16)p1.z, (_Float16)p1.w};
#pragma unroll
                    for (int dt = 0; dt < HD / 16; ++dt) {
                        const pi_u32x4 b = *reinterpret_cast<const pi_u32x4 *>(myvt + ((size_t)(dt * 16 + i) * kAcVtStride + 8 * g) * 2);
                        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa, __builtin_bit_cast(pi_h8, b), acc[dt], 0, 0, 0);
                    }
                }
                issue(vq[u], kt + D3 * kWavesPerBlock);
            }
        }
    }
    // acc[dt][r] = out[token 4g + r][dt*16 + i] over this wave's cells; the four partial tiles meet in wave order
    constexpr int PS = HD + 4;
    float * mypart = reinterpret_cast<float *>(myvt);                                  // [16][PS], inside the wave's own tile
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) mypart[(4 * g + r) * PS + dt * 16 + i] = acc[dt][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * HD; e += kBlock) {
        const int q = e / HD, d = e % HD, t = t0 + q;
        if (t < T) {
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < kWavesPerBlock; ++w) v += reinterpret_cast<const float *>(vt_all + (size_t)w * HD * kAcVtStride * 2)[q * PS + d];
            const size_t o = (size_t)t * out_stride + (size_t)h * HD + d;
            if (q8) {                                  // (a head is whole blocks of 32: half-waves go on together)
                out16[q8 == 2 ? ol_index_of(t, h * HD + d, out_stride) : o] = __float2half_rn(q8_block_value(v));
                continue;
            }
            out[o] = v;
            if (out16) out16[o] = __float2half_rn(v);
        }
    }
}

// ---------------------------------------------------------------------------------------------------
// Attention of a prompt chunk, 64 U tokens of one query head per workgroup.  attn_chunk_mfma_kernel reads a head's cells once for 16
// tokens, holds all their scores in LDS (which ends at about 1850 cells) and is bound by those reads; here a tile of 64 cells is staged
// once for 64 or 128 tokens and no score leaves the registers, so the cells a chunk may see are not limited.  The soft-max keeps the
// rounding points of attn_decode_kernel (fp16 in and out of exp relative to the row's maximum over ALL its cells, e / sum to fp16), which
// is why the keys are gone through three times: for the maximum (products and comparisons only), the sum, and the weights.  Dividing the
// result by the sum instead, in two passes, is a third faster and no further from the exact result, but 2e-4 from the CPU path's: a
// Q4_0 model's next rounding to eight bits then falls the other way for one activation in forty.
// Scores are formed transposed (cells x tokens): a lane's scores belong to one token, and its weights are already the column operand of
// values^T x weights - which cell a slot of that product's inner dimension stands for is free, so the values are read (transposed,
// ds_read_tr16) in the order the scores came out.  A row's sum is exact, whatever the order.
// Bound by the exponentials (about 40 cycles of VALU per 64 of them) beside 48 of matrix cores.  32 heads of 128, RoPE and store included:
// 512 tokens behind 0 / 512 / 1024 / 1535: 43 / 65 / 87 / 110 us (attn_chunk_mfma_kernel 51 / 104 / 145, attn_decode_kernel 700 past the
// cells that one holds), 2046 tokens at once 196 (190 with the sums of 64 weights in float32); 128 heads of 64 on 8: 52 / 98 / 143 / 186
// (75 / 255 / 364 / 479).
// ---------------------------------------------------------------------------------------------------
typedef short pi_s4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ pi_u32x2 lds_tr_read(const unsigned char * q) {
    return __builtin_bit_cast(pi_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pi_s4 *)(__attribute__((address_space(3))) void *)q));
}
constexpr int kRowsCells = 64;                 // cells of a tile
// a soft-max weight (fp16, 0 .. 1) in units of 2^-24; no number counts 0 (the instruction's result, where a C++ conversion has none): its weight
// itself takes it to the output
__device__ __forceinline__ uint32_t weight_units(_Float16 w) {
    uint32_t n;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(n) : "v"((float)w * 16777216.0f));
    return n;
}
template <int HD> constexpr int rows_pitch() { return HD * 2 + 16; }                       // bytes of a staged row: 16 of padding spread the rows over the banks
template <int HD> constexpr size_t rows_lds() { return (size_t)4 * kRowsCells * rows_pitch<HD>(); }

// WHOLE: the weights meet the values before they are divided (e in fp16, the fp32 result divided once), as the parts of attn_part_kernel do, which
// is where decoding goes in caches beyond what attn_decode_kernel holds.  Those round fp16(s - max) by their part's maximum, closer to a
// score than the row's: here s - max stays as it is (40 tokens, 4 heads of 128, 2540 cells, error of the output: four parts 3.6e-4,
// rounded by the row's maximum 4.3e-4).  The keys are then gone through twice: 512 tokens behind 3000, 32 heads of 128: 177 -> 138 us.
template <int HD, int U, bool WHOLE>
__global__ __launch_bounds__(kBlock, 2) void attn_chunk_rows_kernel(const float * __restrict__ q_rot, const __half * __restrict__ k_cache,
                                                                    const __half * __restrict__ v_cache, int n_head, int n_head_kv, int n_ctx,
                                                                    const int32_t * __restrict__ pos_p, int T, int n_kv_max, float * __restrict__ out,
                                                                    int q_stride, int out_stride, __half * __restrict__ out16) {
    static_assert(HD == 128 || HD == 64, "head size");
    constexpr int R = 64 * U, NK = kRowsCells, KS = HD / 32, VT = HD / 16, KT = NK / 16, ROW = rows_pitch<HD>(), PPR = HD / 8, NP = NK * PPR / kBlock;
    extern __shared__ __align__(16) unsigned char smem[];                                  // two tiles of keys, two of values
    __shared__ int span[2 * kWavesPerBlock], odd[2];
    const int h = blockIdx.x, kvh = h / (n_head / n_head_kv), t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * R;      // the tokens that see the most cells first
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
    // the most and the fewest cells a token here sees
    {
        const int t = t0 + tid % R, nv = t < T ? min(pos_p[t] + 1, n_kv_max) : -1;
        int hi = nv, lo = nv < 0 ? INT32_MAX : nv;
        for (int o = 32; o > 0; o >>= 1) { hi = max(hi, __shfl_xor(hi, o, PI_WAVE)); lo = min(lo, __shfl_xor(lo, o, PI_WAVE)); }
        if (lane == 0) { span[wave] = hi; span[kWavesPerBlock + wave] = lo; }
        if (tid < 2) odd[tid] = 0;
    }
    int nv[U];
    pi_u32x4 qf[U][KS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = t0 + wave * 16 * U + u * 16 + i;
        nv[u] = t < T ? min(pos_p[t] + 1, n_kv_max) : 0;
        const float * qp = q_rot + (size_t)min(t, T - 1) * q_stride + (size_t)h * HD + 8 * g;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const float4 a = *reinterpret_cast<const float4 *>(qp + s * 32), b = *reinterpret_cast<const float4 *>(qp + s * 32 + 4);
            qf[u][s] = __builtin_bit_cast(pi_u32x4, pi_h8{(_Float16)a.x, (_Float16)a.y, (_Float16)a.z, (_Float16)a.w, (_Float16)b.x, (_Float16)b.y, (_Float16)b.z, (_Float16)b.w});
        }
    }
    __syncthreads();
    int n_keys = span[0], n_all = span[kWavesPerBlock];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w) { n_keys = max(n_keys, span[w]); n_all = min(n_all, span[kWavesPerBlock + w]); }
    // this thread's pieces of a tile; cells past the last one read the last one again (never a cell that no token here sees)
    const __half * kb = k_cache + (size_t)kvh * n_ctx * HD + (tid % PPR) * 8;
    const __half * vb = v_cache + (size_t)kvh * n_ctx * HD + (tid % PPR) * 8;
    const int row0 = tid / PPR, last = max(n_keys - 1, 0);
    pi_u32x4 pk[NP], pv[NP];
    auto fetch = [&](pi_u32x4 * dst, const __half * base, int cb) {
#pragma unroll
        for (int j = 0; j < NP; ++j) dst[j] = pi_ld16(base + (size_t)min(cb + row0 + j * (kBlock / PPR), last) * HD);
    };
    auto place = [&](unsigned char * tile, const pi_u32x4 * src) {
#pragma unroll
        for (int j = 0; j < NP; ++j) *reinterpret_cast<pi_u32x4 *>(tile + (row0 + j * (kBlock / PPR)) * ROW + (tid % PPR) * 16) = src[j];
    };
    auto products = [&](const unsigned char * tile, pi_f4 (*s)[KT]) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
            for (int u = 0; u < U; ++u) s[u][kt] = pi_f4{0, 0, 0, 0};
#pragma unroll
            for (int c = 0; c < KS; ++c) {
                const pi_u32x4 a = *reinterpret_cast<const pi_u32x4 *>(tile + (kt * 16 + i) * ROW + c * 64 + g * 16);
#pragma unroll
                for (int u = 0; u < U; ++u) s[u][kt] = mma16<__half>(a, qf[u][c], s[u][kt]);
            }
        }
    };
    constexpr int TILE = NK * ROW;
    const float scale = pi_inv_sqrt((float)HD);

    // ---- the rows' maxima (two tiles of keys in LDS: one barrier a tile) ----
    float mx[U];
#pragma unroll
    for (int u = 0; u < U; ++u) mx[u] = -INFINITY;
    int at = 0;
    fetch(pk, kb, 0);
    for (int cb = 0; cb < n_keys; cb += NK, at ^= 1) {
        place(smem + at * TILE, pk);
        __syncthreads();
        fetch(pk, kb, cb + NK);
        pi_f4 s[U][KT];
        products(smem + at * TILE, s);
        const bool edge = cb + NK > n_all;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx[u] = fmaxf(mx[u], edge && cb + kt * 16 + 4 * g + r >= nv[u] ? -INFINITY : s[u][kt][r]);
    }
    float base[U];                                                       // the maximum of the scaled scores
#pragma unroll
    for (int u = 0; u < U; ++u) {
        mx[u] = fmaxf(mx[u], __shfl_xor(mx[u], 16, PI_WAVE));
        mx[u] = fmaxf(mx[u], __shfl_xor(mx[u], 32, PI_WAVE));
        base[u] = mx[u] == -INFINITY ? 0.0f : __fmul_rn(mx[u], scale);
    }

    // e = fp16(exp(fp16(s - max))) of a lane's cells of a tile.  e^x = 2^n 2^(x log2 e - n): log2 e in
    // two parts, so that 2^ is off by little more than its own rounding
    auto weigh = [&](const pi_f4 * s, int cb, bool edge, int seen, float b, _Float16 * w) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float d = __fsub_rn(__fmul_rn(s[kt][r], scale), b), x = WHOLE ? d : (float)(_Float16)d;
                const float n = fmaxf(__builtin_rintf(x * 1.44269504f), -200.0f);                // x may be -inf
                const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(fmaf(x, 1.92596303e-08f, fmaf(x, 1.44269502f, -n))), (int)n);
                w[kt * 4 + r] = (_Float16)(edge && cb + kt * 16 + 4 * g + r >= seen ? 0.0f : e);
            }
    };

    // ---- the rows' sums, exact as the CPU path's sums in double are: a weight is a whole number of 2^-24, of which a lane adds 16 a tile ----
    double sum[U];
#pragma unroll
    for (int u = 0; u < U; ++u) sum[u] = 0.0;
    auto add_weights = [&](const _Float16 * w, double & to) {
        uint32_t part = 0;                                               // at most 2^28
#pragma unroll
        for (int k = 0; k < 4 * KT; ++k) part += weight_units(w[k]);
        to += (double)part;
    };
    auto total = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            sum[u] += __shfl_xor(sum[u], 16, PI_WAVE);
            sum[u] += __shfl_xor(sum[u], 32, PI_WAVE);
            sum[u] *= 5.9604644775390625e-08;                            // 2^-24
        }
    };
    if constexpr (!WHOLE) {
        fetch(pk, kb, 0);
        __syncthreads();                                                 // the last tile of the pass before has been read
        at = 0;
        for (int cb = 0; cb < n_keys; cb += NK, at ^= 1) {
            place(smem + at * TILE, pk);
            __syncthreads();
            fetch(pk, kb, cb + NK);
            pi_f4 s[U][KT];
            products(smem + at * TILE, s);
            const bool edge = cb + NK > n_all;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                _Float16 w[4 * KT];
                weigh(s[u], cb, edge, nv[u], base[u], w);
                add_weights(w, sum[u]);
            }
        }
        total();
    }

    // ---- weights and values ----
    float inv[U];
    pi_f4 o[U][VT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        inv[u] = WHOLE ? 1.0f : (float)(1.0 / sum[u]);
#pragma unroll
        for (int v = 0; v < VT; ++v) o[u][v] = pi_f4{0, 0, 0, 0};
    }
    unsigned char * vt = smem + 2 * TILE;
    fetch(pk, kb, 0);
    fetch(pv, vb, 0);
    __syncthreads();
    at = 0;
    for (int cb = 0; cb < n_keys; cb += NK, at ^= 1) {
        const bool edge = cb + NK > n_all;
        place(smem + at * TILE, pk);
        place(vt + at * TILE, pv);
        if (edge) {                                                      // a value that is no number, in a cell that some tokens here do not see
            unsigned bad = 0;
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int w = 0; w < 4; ++w) { const unsigned x = pv[j][w] & 0x7C007C00u; bad |= (x & 0xFFFFu) == 0x7C00u || (x >> 16) == 0x7C00u; }
            if (bad) odd[at] = 1;
        }
        __syncthreads();
        fetch(pk, kb, cb + NK);
        fetch(pv, vb, cb + NK);
        pi_f4 s[U][KT];
        products(smem + at * TILE, s);
        pi_u32x4 pb[U][KT / 2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            _Float16 w[4 * KT];
            weigh(s[u], cb, edge, nv[u], base[u], w);
            if constexpr (WHOLE) add_weights(w, sum[u]);
            else {
#pragma unroll
                for (int k = 0; k < 4 * KT; ++k) w[k] = (_Float16)__fmul_rn((float)w[k], inv[u]);
            }
#pragma unroll
            for (int k = 0; k < KT / 2; ++k)
                pb[u][k] = __builtin_bit_cast(pi_u32x4, pi_h8{w[k * 8], w[k * 8 + 1], w[k * 8 + 2], w[k * 8 + 3], w[k * 8 + 4], w[k * 8 + 5], w[k * 8 + 6], w[k * 8 + 7]});
        }
        const unsigned char * vs = vt + at * TILE;
        if (edge && odd[at]) {
            // 0 times such a value is no number either: token by token, the cells it sees only.  The weight of cell (kt, g, r) of token i is
            // half (kt % 2) * 4 + r of step kt / 2 in lane 16 g + i.
#pragma unroll
            for (int u = 0; u < U; ++u)
                for (int c = 0; c < NK; ++c) {
                    const int kt = c >> 4, from = ((c >> 2) & 3) * 16 + i, half = (kt & 1) * 4 + (c & 3);
                    unsigned word = 0;
#pragma unroll
                    for (int k = 0; k < KT / 2; ++k)
#pragma unroll
                        for (int q = 0; q < 4; ++q) word = k == (kt >> 1) && q == (half >> 1) ? pb[u][k][q] : word;
                    const unsigned got = (unsigned)__shfl((int)word, from, PI_WAVE);
                    const float w = pi_f16_from_bits((uint16_t)(half & 1 ? got >> 16 : got));
                    if (cb + c >= nv[u]) continue;
#pragma unroll
                    for (int v = 0; v < VT; ++v)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[u][v][r] = fmaf(w, __half2float(reinterpret_cast<const __half *>(vs + c * ROW)[v * 16 + 4 * g + r]), o[u][v][r]);
                }
            continue;
        }
        // slot (g, j) of a 32-cell step: cell 4 g + j of its first 16 (j < 4) or of its second 16 - two transposing reads
#pragma unroll
        for (int k = 0; k < KT / 2; ++k)
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const unsigned char * a = vs + (k * 32 + 4 * g + (i >> 2)) * ROW + (v * 16 + (i & 3) * 4) * 2;
                const pi_u32x2 lo = lds_tr_read(a), hi = lds_tr_read(a + 16 * ROW);
                const pi_u32x4 fr{lo.x, lo.y, hi.x, hi.y};
#pragma unroll
                for (int u = 0; u < U; ++u) o[u][v] = mma16<__half>(fr, pb[u][k], o[u][v]);
            }
    }
    if constexpr (WHOLE) total();
    // o[u][v][r] = out[token i][v * 16 + 4 g + r]
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = t0 + wave * 16 * U + u * 16 + i;
        if (t >= T) continue;
        float * po = out + (size_t)t * out_stride + (size_t)h * HD + 4 * g;
        __half * ph = out16 ? out16 + (size_t)t * out_stride + (size_t)h * HD + 4 * g : nullptr;
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            float4 y{o[u][v][0], o[u][v][1], o[u][v][2], o[u][v][3]};
            if constexpr (WHOLE) { const float d = (float)sum[u]; y = float4{pi_div(y.x, d), pi_div(y.y, d), pi_div(y.z, d), pi_div(y.w, d)}; }
            *reinterpret_cast<float4 *>(po + v * 16) = y;
            if (ph) {
                typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<h4 *>(ph + v * 16) = h4{(_Float16)y.x, (_Float16)y.y, (_Float16)y.z, (_Float16)y.w};
            }
        }
    }
}

// The same 64 U tokens of a head against their cells in ONE pass over the keys: weights relative to a maximum that grows as the cells come, values
// under the undivided weights (fp16), one division at the end.  For models of F16 matrices, whose next rounding is to fp16: against the three passes
// above the result has two roundings fewer a weight (of s - max and of e / sum), and no eight-bit step behind it that a last place could turn.
// A row's base is raised only where a score exceeds it by more than 2^8 (weights up to 256 in fp16, the sums in their wider types): then what
// has been added so far is scaled down, which is rare, and no lane needs its neighbours' maxima to know that it is not needed.
// The weights' sum is a product too (with ones, exact products of the same fp16 weights), a tile of 64 cells at a time, added up in double.
// Bound by LDS (a tile's keys and values pass to each of four waves: about as many cycles as its products) and the exponentials between the two products.
// RoPE and store included, three passes / one: 32 heads of 128, 2046 tokens 200 / 80 us, 512 42 / 25, 512 behind 1024 87 / 42, 64 15.0 / 11.7; 128
// heads of 64 on 8, 1900 tokens 323 / 105; error against float64 (2046 tokens) 3.9e-4 / 2.6e-4.
template <int HD, int U>
__global__ __launch_bounds__(kBlock, 2) void attn_chunk_rows_once_kernel(const __half * __restrict__ q16, const __half * __restrict__ k_cache, const __half * __restrict__ v_cache,
                                                                         int n_head, int n_head_kv, int n_ctx, const int32_t * __restrict__ pos_p, int T, int n_kv_max, int fold,
                                                                         float * __restrict__ out, int out_stride, __half * __restrict__ out16) {
    static_assert(HD == 128 || HD == 64, "head size");
    constexpr int R = 64 * U, NK = kRowsCells, KS = HD / 32, VT = HD / 16, KT = NK / 16, ROW = rows_pitch<HD>(), PPR = HD / 8, NP = NK * PPR / kBlock;
    extern __shared__ __align__(16) unsigned char smem[];                                  // two tiles of keys, two of values
    __shared__ int span[2 * kWavesPerBlock], odd[2];
    // the tokens that see the most cells first; where all workgroups run at once (fold) the second half of them the other way round, so that a
    // unit's two have the same number of cells together
    const int nb = (int)gridDim.y, y = (int)blockIdx.y, half = (nb + 1) / 2, tb = fold && y >= half ? y - half : nb - 1 - y;
    const int h = blockIdx.x, kvh = h / (n_head / n_head_kv), t0 = tb * R;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
    // the most and the fewest cells a token here sees
    {
        const int t = t0 + tid % R, nv = t < T ? min(pos_p[t] + 1, n_kv_max) : -1;
        int hi = nv, lo = nv < 0 ? INT32_MAX : nv;
        for (int o = 32; o > 0; o >>= 1) { hi = max(hi, __shfl_xor(hi, o, PI_WAVE)); lo = min(lo, __shfl_xor(lo, o, PI_WAVE)); }
        if (lane == 0) { span[wave] = hi; span[kWavesPerBlock + wave] = lo; }
        if (tid < 2) odd[tid] = 0;
    }
    int nv[U];
    pi_u32x4 qf[U][KS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = t0 + wave * 16 * U + u * 16 + i;
        nv[u] = t < T ? min(pos_p[t] + 1, n_kv_max) : 0;
        const __half * qp = q16 + ((size_t)min(t, T - 1) * n_head + h) * HD + 8 * g;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[u][s] = pi_ld16(qp + s * 32);
    }
    __syncthreads();
    int n_keys = span[0], n_all = span[kWavesPerBlock];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w) { n_keys = max(n_keys, span[w]); n_all = min(n_all, span[kWavesPerBlock + w]); }
    // this thread's pieces of a tile; cells past the last one read the last one again (never a cell that no token here sees)
    const __half * kb = k_cache + (size_t)kvh * n_ctx * HD + (tid % PPR) * 8;
    const __half * vb = v_cache + (size_t)kvh * n_ctx * HD + (tid % PPR) * 8;
    const int row0 = tid / PPR, last = max(n_keys - 1, 0);
    pi_u32x4 pk[NP], pv[NP];
    auto fetch = [&](pi_u32x4 * dst, const __half * base, int cb) {
#pragma unroll
        for (int j = 0; j < NP; ++j) dst[j] = pi_ld16(base + (size_t)min(cb + row0 + j * (kBlock / PPR), last) * HD);
    };
    auto place = [&](unsigned char * tile, const pi_u32x4 * src) {
#pragma unroll
        for (int j = 0; j < NP; ++j) *reinterpret_cast<pi_u32x4 *>(tile + (row0 + j * (kBlock / PPR)) * ROW + (tid % PPR) * 16) = src[j];
    };
    constexpr int TILE = NK * ROW;
    const float to2 = pi_inv_sqrt((float)HD) * 1.44269504f, room = 8.0f / to2;             // e^(s / sqrt(HD)) = 2^(s to2)
    const pi_u32x4 ones{0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};

    float limit[U], base2[U];                                            // a score beyond it raises the base; the base as a power of two (0 while there is none)
    double sum[U];
    pi_f4 o[U][VT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        limit[u] = -INFINITY; base2[u] = 0.0f; sum[u] = 0.0;
#pragma unroll
        for (int v = 0; v < VT; ++v) o[u][v] = pi_f4{0, 0, 0, 0};
    }
    unsigned char * vt = smem + 2 * TILE;
    fetch(pk, kb, 0);
    fetch(pv, vb, 0);
    int at = 0;
    for (int cb = 0; cb < n_keys; cb += NK, at ^= 1) {
        const bool edge = cb + NK > n_all;
        place(smem + at * TILE, pk);
        place(vt + at * TILE, pv);
        if (edge) {                                                      // a value that is no number, in a cell that some tokens here do not see
            unsigned bad = 0;
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int w = 0; w < 4; ++w) { const unsigned x = pv[j][w] & 0x7C007C00u; bad |= (x & 0xFFFFu) == 0x7C00u || (x >> 16) == 0x7C00u; }
            if (bad) odd[at] = 1;
        }
        __syncthreads();
        fetch(pk, kb, cb + NK);
        fetch(pv, vb, cb + NK);
        pi_f4 s[U][KT];
        const unsigned char * tile = smem + at * TILE;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
            for (int u = 0; u < U; ++u) s[u][kt] = pi_f4{0, 0, 0, 0};
#pragma unroll
            for (int c = 0; c < KS; ++c) {
                const pi_u32x4 a = *reinterpret_cast<const pi_u32x4 *>(tile + (kt * 16 + i) * ROW + c * 64 + g * 16);
#pragma unroll
                for (int u = 0; u < U; ++u) s[u][kt] = mma16<__half>(a, qf[u][c], s[u][kt]);
            }
        }
        if (edge) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[u][kt][r] = cb + kt * 16 + 4 * g + r >= nv[u] ? -INFINITY : s[u][kt][r];
        }
        pi_u32x4 pb[U][KT / 2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float top = s[u][0][0];
#pragma unroll
            for (int k = 1; k < 4 * KT; ++k) top = fmaxf(top, s[u][k >> 2][k & 3]);
            if (__any(top > limit[u])) {
                top = fmaxf(top, __shfl_xor(top, 16, PI_WAVE));
                top = fmaxf(top, __shfl_xor(top, 32, PI_WAVE));
                if (top > limit[u] - room) {                             // (limit -inf: -inf)
                    const float b = top * to2, down = limit[u] == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(base2[u] - b);
                    limit[u] = top + room; base2[u] = b;
                    sum[u] *= (double)down;
#pragma unroll
                    for (int v = 0; v < VT; ++v) o[u][v] *= down;
                }
            }
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
            typedef float f2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int k = 0; k < 2 * KT; ++k) {
                const f2 e{__builtin_amdgcn_exp2f(fmaf(s[u][k >> 1][2 * (k & 1)], to2, -base2[u])), __builtin_amdgcn_exp2f(fmaf(s[u][k >> 1][2 * (k & 1) + 1], to2, -base2[u]))};
                pb[u][k >> 2][k & 3] = __builtin_bit_cast(unsigned, __builtin_convertvector(e, h2));
            }
            pi_f4 n{0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < KT / 2; ++k) n = mma16<__half>(ones, pb[u][k], n);
            sum[u] += (double)n[0];
        }
        const unsigned char * vs = vt + at * TILE;
        if (edge && odd[at]) {
            // 0 times such a value is no number either: token by token, the cells it sees only.  The weight of cell (kt, g, r) of token i is
            // half (kt % 2) * 4 + r of step kt / 2 in lane 16 g + i.
#pragma unroll
            for (int u = 0; u < U; ++u)
                for (int c = 0; c < NK; ++c) {
                    const int kt = c >> 4, from = ((c >> 2) & 3) * 16 + i, hw = (kt & 1) * 4 + (c & 3);
                    unsigned word = 0;
#pragma unroll
                    for (int k = 0; k < KT / 2; ++k)
#pragma unroll
                        for (int q = 0; q < 4; ++q) word = k == (kt >> 1) && q == (hw >> 1) ? pb[u][k][q] : word;
                    const unsigned got = (unsigned)__shfl((int)word, from, PI_WAVE);
                    const float w = pi_f16_from_bits((uint16_t)(hw & 1 ? got >> 16 : got));
                    if (cb + c >= nv[u]) continue;
#pragma unroll
                    for (int v = 0; v < VT; ++v)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[u][v][r] = fmaf(w, __half2float(reinterpret_cast<const __half *>(vs + c * ROW)[v * 16 + 4 * g + r]), o[u][v][r]);
                }
            continue;
        }
        // slot (g, j) of a 32-cell step: cell 4 g + j of its first 16 (j < 4) or of its second 16 - two transposing reads
#pragma unroll
        for (int k = 0; k < KT / 2; ++k)
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const unsigned char * a = vs + (k * 32 + 4 * g + (i >> 2)) * ROW + (v * 16 + (i & 3) * 4) * 2;
                const pi_u32x2 lo = lds_tr_read(a), hi = lds_tr_read(a + 16 * ROW);
                const pi_u32x4 fr{lo.x, lo.y, hi.x, hi.y};
#pragma unroll
                for (int u = 0; u < U; ++u) o[u][v] = mma16<__half>(fr, pb[u][k], o[u][v]);
            }
    }
    // o[u][v][r] = out[token i][v * 16 + 4 g + r]
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = t0 + wave * 16 * U + u * 16 + i;
        if (t >= T) continue;
        const float inv = (float)(1.0 / sum[u]);
        const size_t to = (size_t)t * out_stride + (size_t)h * HD + 4 * g;
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            const float4 y{o[u][v][0] * inv, o[u][v][1] * inv, o[u][v][2] * inv, o[u][v][3] * inv};
            if (out) *reinterpret_cast<float4 *>(out + to + v * 16) = y;
            if (out16) {
                typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<h4 *>(out16 + to + v * 16) = h4{(_Float16)y.x, (_Float16)y.y, (_Float16)y.z, (_Float16)y.w};
            }
        }
    }
}

// RoPE + KV store of a chunk's tokens, all heads of a token by one workgroup (or by gridDim.y of them, heads in turn): the angles are
// formed once a token instead of once a head, bit for bit those of rope_kv_store_kernel, and the rest is a copy at the rate of memory.
__global__ __launch_bounds__(kBlock) void rope_kv_chunk_kernel(const float * __restrict__ qkv, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                                                               const int32_t * __restrict__ pos_p, int n_ctx, float * __restrict__ q_rot,
                                                               __half * __restrict__ k_cache, __half * __restrict__ v_cache, int qkv_stride, int q_stride) {
    extern __shared__ __align__(16) unsigned char smem[];
    float2 * cs = reinterpret_cast<float2 *>(smem);                      // [hd / 2]
    const int t = blockIdx.x, tid = threadIdx.x, half = hd / 2, pos = pos_p[t];
    for (int j = tid; j < half; j += kBlock) {
        const float theta = rope_angle((float)pos, j, mode, theta_scale, freq_scale);
        cs[j] = make_float2(cosf(theta), sinf(theta));
    }
    __syncthreads();
    const float * src = qkv + (size_t)t * qkv_stride;
    float * qd = q_rot + (size_t)t * q_stride;
    const int pairs = (n_head + 2 * n_head_kv) * half;
    for (int e = blockIdx.y * kBlock + tid; e < pairs; e += gridDim.y * kBlock) {
        const int h = e / half, j = e % half;
        const bool value = h >= n_head + n_head_kv;
        const int i0 = (mode & 2) && !value ? j : 2 * j, i1 = (mode & 2) && !value ? j + half : 2 * j + 1;
        const float x0 = src[(size_t)h * hd + i0], x1 = src[(size_t)h * hd + i1];
        if (value) {
            __half * dst = v_cache + ((size_t)(h - n_head - n_head_kv) * n_ctx + pos) * hd;
            dst[i0] = __float2half_rn(x0); dst[i1] = __float2half_rn(x1);
            continue;
        }
        const float c = cs[j].x, s = cs[j].y;
        const float y0 = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, s)), y1 = __fadd_rn(__fmul_rn(x0, s), __fmul_rn(x1, c));
        if (h < n_head) {
            qd[(size_t)h * hd + i0] = y0; qd[(size_t)h * hd + i1] = y1;
        } else {
            __half * dst = k_cache + ((size_t)(h - n_head) * n_ctx + pos) * hd;
            dst[i0] = __float2half_rn(y0); dst[i1] = __float2half_rn(y1);
        }
    }
}

// The same where rows and heads allow 16-byte accesses: a thread has eight values of a head (neighbours, or four and the four they rotate with), requested
// before the angles are formed, and a workgroup 256 such pieces of a token.  Bound by the trip there and back in short chunks, by the copy in long
// ones (167 MB in and out of 2046 tokens).  The angles of a token are formed once a workgroup, which costs less than more pieces of a thread one after the other do: 32
// heads of 128, a workgroup of a token (four up to 511 tokens, sixteen up to 127) with up to six pieces a thread in flight / this, us: 21 tokens 5.0 / 4.2, 130 6.6 / 5.7,
// 300 8.3 / 7.0, 508 12.3 / 10.0; queries in fp16, 508 12.9 / 10.2, 999 15.6 / 15.9, 2046 29.4 / 28.4.
// Q16: the rotated queries leave rounded to fp16, rows of n_head * hd of them (what attn_chunk_rows_once_kernel reads: half the bytes of both launches).
template <bool Q16>
__global__ __launch_bounds__(kBlock) void rope_kv_chunk_wide_kernel(const float * __restrict__ qkv, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                                                                     const int32_t * __restrict__ pos_p, int n_ctx, float * __restrict__ q_rot,
                                                                     __half * __restrict__ k_cache, __half * __restrict__ v_cache, int qkv_stride, int q_stride) {
    extern __shared__ __align__(16) unsigned char smem[];
    float2 * cs = reinterpret_cast<float2 *>(smem);                      // [hd / 2]
    const int t = blockIdx.x, tid = threadIdx.x, half = hd / 2, pos = pos_p[t], per = hd / 8, n = (n_head + 2 * n_head_kv) * per;
    const float * src = qkv + (size_t)t * qkv_stride;
    float * qd = q_rot + (size_t)t * q_stride;
    const bool neox = (mode & 2) != 0;
    const int step = neox ? 4 : 8, second = neox ? half : 4;             // of a piece: where it starts in the head (times its number), where its second four are
    const int e = min((int)blockIdx.y * kBlock + tid, n - 1), h = e / per, j = e % per;     // (past the end the last piece again, not stored)
    const float4 a = *reinterpret_cast<const float4 *>(src + (size_t)h * hd + j * step), b = *reinterpret_cast<const float4 *>(src + (size_t)h * hd + j * step + second);
    for (int k = tid; k < half; k += kBlock) {
        const float theta = rope_angle((float)pos, k, mode, theta_scale, freq_scale);
        cs[k] = make_float2(cosf(theta), sinf(theta));
    }
    __syncthreads();
    if ((int)blockIdx.y * kBlock + tid >= n) return;
    float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    if (h < n_head + n_head_kv) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float & x0 = neox ? x[q] : x[2 * q], & x1 = neox ? x[q + 4] : x[2 * q + 1];
            const float2 w = cs[4 * j + q];
            const float y0 = __fsub_rn(__fmul_rn(x0, w.x), __fmul_rn(x1, w.y)), y1 = __fadd_rn(__fmul_rn(x0, w.y), __fmul_rn(x1, w.x));
            x0 = y0; x1 = y1;
        }
    }
    if (!Q16 && h < n_head) {
        float * dst = qd + (size_t)h * hd + j * step;
        *reinterpret_cast<float4 *>(dst) = make_float4(x[0], x[1], x[2], x[3]);
        *reinterpret_cast<float4 *>(dst + second) = make_float4(x[4], x[5], x[6], x[7]);
    } else {
        const int hk = h - n_head;
        __half * dst = (h < n_head ? reinterpret_cast<__half *>(q_rot) + (size_t)t * q_stride + (size_t)h * hd
                        : hk < n_head_kv ? k_cache + ((size_t)hk * n_ctx + pos) * hd : v_cache + ((size_t)(hk - n_head_kv) * n_ctx + pos) * hd) + j * step;
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<h4 *>(dst) = h4{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]};
        *reinterpret_cast<h4 *>(dst + second) = h4{(_Float16)x[4], (_Float16)x[5], (_Float16)x[6], (_Float16)x[7]};
    }
}

// ---------------------------------------------------------------------------------------------------
// One token's attention on the layouts of the reference's own KV cache (llm_build_kv_store / llm_build_kqv, llama.cpp:4383-4418,
// 4764-4850): K cells [cell][n_head_kv * hd] fp16, V transposed [n_head_kv * hd][n_ctx] fp16.  What its graph spreads over eleven nodes
// - RoPE of q and k, the two copies into the cache, K.q, scale, + mask, soft-max, V.p and the gather of the heads - is one launch, one
// workgroup per query head, with the CPU path's rounding points: q and p rounded to fp16 in front of their products (the mat-muls
// against fp16 operands, ggml.c:9703-9716), exp through fp16 on both sides (ggml.c:10747-10759), the sum of the exponentials in double.
// The new cell's K and V rows are used from LDS (every head of a group computes them, the group's first head stores them), so no
// workgroup depends on another's stores.  Cells whose mask entry is -inf get probability 0 whatever the cache holds there.
// RoPE as rope_kernel of the boundary computes it: angle advanced by repeated fp32 multiplication, cosf / sinf, * mscale.
// ---------------------------------------------------------------------------------------------------
// A step of T tokens (grid.y; token u's q, k, v at stride tok_stride, its cell cell0 + u, its mask row at mask_stride, its output at
// out_stride): the K and V rows of all T new cells are formed in LDS by every workgroup, so a token attends the other tokens of its
// step (where its mask allows) without waiting for their stores - what the reference gets by storing the whole batch first.
__global__ __launch_bounds__(kBlock) void attn_ggml_kernel(const float * __restrict__ q, const float * __restrict__ k, const float * __restrict__ v, int tok_stride,
                                                           const int32_t * __restrict__ pos, int mode, float theta_scale, float freq_scale, float mscale,
                                                           __half * __restrict__ k_cache, __half * __restrict__ v_cache,
                                                           int n_head, int n_head_kv, int hd, int n_ctx, int n_kv, int T, int cell0,
                                                           const float * __restrict__ kq_scale, const float * __restrict__ kq_mask, int mask_stride,
                                                           float * __restrict__ out, int out_stride) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n_kv8 = (n_kv + 7) & ~7;                                     // the V rows are read eight cells at a time
    float * sc = reinterpret_cast<float *>(smem);                          // [n_kv8] scores, then probabilities (zeros behind n_kv)
    __half * q16 = reinterpret_cast<__half *>(sc + n_kv8);                 // [hd]
    __half * k16 = q16 + hd;                                               // [T][hd] the step's new K rows
    __half * v16 = k16 + (size_t)T * hd;                                   // [T][hd] and V rows
    __shared__ double red[kWavesPerBlock];
    __shared__ float  redf[kWavesPerBlock];
    const int h = blockIdx.x, tok = blockIdx.y, kvh = h / (n_head / n_head_kv), gqa = n_head_kv * hd;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool owner = h % (n_head / n_head_kv) == 0;                      // this head's workgroup stores the group's new K / V rows of its token
    const int cell = cell0 + tok;
    kq_mask += (size_t)tok * mask_stride;
    out += (size_t)tok * out_stride;
    if (tid < hd / 2) {
        const int i = tid;
        const int i0 = (mode & 2) ? i : 2 * i, i1 = (mode & 2) ? i + hd / 2 : 2 * i + 1;
        for (int u = 0; u < T; ++u) {
            float theta = (float)pos[u];
            if (mode & 2) theta = __fmul_rn(theta, freq_scale);
            for (int j = 0; j < i; ++j) theta = __fmul_rn(theta, theta_scale);
            const float th = __fmul_rn(freq_scale, theta);
            const float c = __fmul_rn(cosf(th), mscale), sn = __fmul_rn(sinf(th), mscale);
            if (u == tok) {
                const float q0 = q[(size_t)u * tok_stride + h * hd + i0], q1 = q[(size_t)u * tok_stride + h * hd + i1];
                q16[i0] = __float2half_rn(__fsub_rn(__fmul_rn(q0, c), __fmul_rn(q1, sn)));
                q16[i1] = __float2half_rn(__fadd_rn(__fmul_rn(q0, sn), __fmul_rn(q1, c)));
            }
            const float k0 = k[(size_t)u * tok_stride + kvh * hd + i0], k1 = k[(size_t)u * tok_stride + kvh * hd + i1];
            const __half r0 = __float2half_rn(__fsub_rn(__fmul_rn(k0, c), __fmul_rn(k1, sn)));
            const __half r1 = __float2half_rn(__fadd_rn(__fmul_rn(k0, sn), __fmul_rn(k1, c)));
            k16[u * hd + i0] = r0; k16[u * hd + i1] = r1;
            if (owner && u == tok) { k_cache[(size_t)cell * gqa + kvh * hd + i0] = r0; k_cache[(size_t)cell * gqa + kvh * hd + i1] = r1; }
        }
    }
    if (tid < hd) {
        for (int u = 0; u < T; ++u) {
            const __half r = __float2half_rn(v[(size_t)u * tok_stride + kvh * hd + tid]);
            v16[u * hd + tid] = r;
            if (owner && u == tok) v_cache[(size_t)(kvh * hd + tid) * n_ctx + cell] = r;
        }
    }
    __syncthreads();

    // ---- scores: hd / 8 lanes per cell, 16 bytes of the cell's row each; four cells' rows in flight per lane -----------------
    const int lpc = hd / 8, cpw = PI_WAVE / lpc;                          // lanes per cell, cells per wave and pass
    const int sub = lane / lpc, l = lane % lpc;
    const pi_u32x4 qv = *reinterpret_cast<const pi_u32x4 *>(q16 + l * 8);
    const float scale = kq_scale[0];
    constexpr int SU = 4;
    const int cstep = kWavesPerBlock * cpw;
    for (int c0 = wave * cpw + sub; c0 < n_kv; c0 += SU * cstep) {
        pi_u32x4 kr[SU];
        float m[SU];
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const int c = c0 + u * cstep;
            const int cc = c < n_kv ? c : n_kv - 1;                          // (clamped requests keep the loads unconditional)
            m[u] = kq_mask[cc];
            kr[u] = pi_ld16(k_cache + (size_t)cc * gqa + kvh * hd + l * 8);
        }
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const int c = c0 + u * cstep;
            if (c >= cell0 && c < cell0 + T) kr[u] = *reinterpret_cast<const pi_u32x4 *>(k16 + (c - cell0) * hd + l * 8);
            float d = pi_dot8h(kr[u], qv, 0.0f);
            for (int o = 1; o < lpc; o <<= 1) d += __shfl_xor(d, o, PI_WAVE);
            if (c < n_kv && l == 0) sc[c] = m[u] == -INFINITY ? -INFINITY : __fadd_rn(__fmul_rn(d, scale), m[u]);
        }
    }
    __syncthreads();
    // ---- soft-max over the cells -------------------------------------------------------------------------------------------
    float mx = -INFINITY;
    for (int c = tid; c < n_kv; c += kBlock) mx = fmaxf(mx, sc[c]);
    mx = pi_wave_max(mx);
    if (lane == 0) redf[wave] = mx;
    __syncthreads();
    mx = redf[0];
    for (int w = 1; w < kWavesPerBlock; ++w) mx = fmaxf(mx, redf[w]);
    double sum = 0.0;
    for (int c = tid; c < n_kv; c += kBlock) {
        const float e = sc[c] == -INFINITY ? 0.0f : pi_round_f16(expf(pi_round_f16(__fsub_rn(sc[c], mx))));
        sc[c] = e; sum += (double)e;
    }
    sum = pi_wave_sum_f64(sum);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < kWavesPerBlock; ++w) tot += red[w];
    const float inv = (float)(1.0 / tot);
    for (int c = tid; c < n_kv8; c += kBlock) sc[c] = c < n_kv ? __fmul_rn(sc[c], inv) : 0.0f;
    __syncthreads();
    // ---- out[dim] = sum over cells of fp16(p[cell]) * V[dim][cell].  Thread t owns column t % hd and every (kBlock / hd)-th group of
    // eight cells of it, four groups in flight; the column's partial sums meet in LDS (the scores' first floats are free by then
    // only after everyone has read its probabilities, hence the barrier in between) ------------------------------------------------
    {
        const int dim = tid % hd, part = tid / hd, nparts = kBlock / hd;      // hd <= kBlock and divides it (the launcher's test)
        const __half * vr = v_cache + (size_t)(kvh * hd + dim) * n_ctx;
        float acc = 0.0f;
        constexpr int VU = 4;
        for (int g0 = part; g0 * 8 < n_kv; g0 += VU * nparts) {
            pi_u32x4 vv[VU];
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                const int c0 = (g0 + u * nparts) * 8;
                vv[u] = pi_ld16(vr + (c0 < n_kv ? c0 : 0));
            }
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                const int c0 = (g0 + u * nparts) * 8;
                if (c0 < n_kv) {
                    for (int w = c0 > cell0 ? c0 - cell0 : 0; w < T && cell0 + w < c0 + 8; ++w)      // the step's own cells come from LDS
                        reinterpret_cast<__half *>(&vv[u])[cell0 + w - c0] = v16[w * hd + dim];
                    const float4 p0 = *reinterpret_cast<const float4 *>(sc + c0), p1 = *reinterpret_cast<const float4 *>(sc + c0 + 4);
                    __half2 ph[4] = {__floats2half2_rn(p0.x, p0.y), __floats2half2_rn(p0.z, p0.w), __floats2half2_rn(p1.x, p1.y), __floats2half2_rn(p1.z, p1.w)};
                    // a cell without probability contributes nothing, whatever its (possibly never written) V entry holds
                    const uint32_t * pw = reinterpret_cast<const uint32_t *>(ph);
                    uint32_t * vw = reinterpret_cast<uint32_t *>(&vv[u]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if ((pw[j] & 0x0000ffffu) == 0u) vw[j] &= 0xffff0000u;
                        if ((pw[j] & 0xffff0000u) == 0u) vw[j] &= 0x0000ffffu;
                    }
                    acc = pi_dot8h(vv[u], *reinterpret_cast<const pi_u32x4 *>(ph), acc);
                }
            }
        }
        float * pacc = reinterpret_cast<float *>(v16 + (size_t)T * hd);       // [kBlock] floats behind the fp16 rows
        pacc[tid] = acc;
        __syncthreads();
        if (tid < hd) {
            float t = pacc[tid];
            for (int w = 1; w < nparts; ++w) t += pacc[tid + w * hd];
            out[h * hd + tid] = t;
        }
    }
}

}  // namespace

namespace {
constexpr size_t kChunkMfmaLds = 156 * 1024;
size_t chunk_mfma_lds(int hd, int n_kv_max) { return sizeof(float) * 16 * (size_t)(((n_kv_max + 31) & ~31) + 4) + (size_t)kWavesPerBlock * hd * kAcVtStride * 2; }

template <int HD, int U, bool WHOLE>
int launch_chunk_rows(const float * q_rot, const void * k_cache, const void * v_cache, int n_head, int n_head_kv, int n_ctx, const int32_t * pos, int T, int n_kv_max, float * out,
                      int out_stride, void * out_f16, hipStream_t st) {
    static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&attn_chunk_rows_kernel<HD, U, WHOLE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_lds<HD>());
    if (raised != hipSuccess) return pi::hip_fail(raised, "attn_chunk_rows: LDS size");
    hipLaunchKernelGGL((attn_chunk_rows_kernel<HD, U, WHOLE>), dim3(n_head, (T + 64 * U - 1) / (64 * U)), dim3(kBlock), rows_lds<HD>(), st, q_rot, (const __half *)k_cache, (const __half *)v_cache,
                       n_head, n_head_kv, n_ctx, pos, T, n_kv_max, out, n_head * HD, out_stride, (__half *)out_f16);
    return pi::check_launch("attn_chunk_rows");
}
template <int HD, int U>
int launch_chunk_once(const void * q16, const void * k_cache, const void * v_cache, int n_head, int n_head_kv, int n_ctx, const int32_t * pos, int T, int n_kv_max, float * out, int out_stride,
                      void * out_f16, hipStream_t st) {
    static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&attn_chunk_rows_once_kernel<HD, U>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_lds<HD>());
    if (raised != hipSuccess) return pi::hip_fail(raised, "attn_chunk_once: LDS size");
    const int blocks = (T + 64 * U - 1) / (64 * U);
    hipLaunchKernelGGL((attn_chunk_rows_once_kernel<HD, U>), dim3(n_head, blocks), dim3(kBlock), rows_lds<HD>(), st, (const __half *)q16, (const __half *)k_cache, (const __half *)v_cache,
                       n_head, n_head_kv, n_ctx, pos, T, n_kv_max, (long long)n_head * blocks <= 2 * pi::compute_units() ? 1 : 0, out, out_stride, (__half *)out_f16);
    return pi::check_launch("attn_chunk_once");
}
}  // namespace

namespace pi {
// keys and values of T tokens to their cells, rotated queries to q_rot; n_head 0: rows of k and v alone (no q_rot)
int rope_kv_chunk(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale, const int32_t * pos, int n_ctx,
                  float * q_rot, void * k_cache, void * v_cache, hipStream_t st, bool q16) {
    // 16 tokens and fewer: a workgroup per head and token (16 tokens, 32 heads of 128, attention included: 11.8 against 12.3 us); a chunk's angles
    // are worth forming less often from there on.  Other rows: a workgroup per token fills the chip from 512 tokens; shorter chunks split its heads
    if (T <= kBtMaxT) {
        hipLaunchKernelGGL(rope_kv_store_kernel, dim3(n_head + 2 * n_head_kv, T), dim3(hd / 2), 0, st,
                           qkv, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, q_rot, (__half *)k_cache, (__half *)v_cache, qkv_stride, n_head * hd);
        return pi::check_launch("rope_kv_store");
    }
    // 16-byte rows: heads of a multiple of eight values, and everything that starts on one
    const bool wide = hd % 8 == 0 && qkv_stride % 4 == 0 && (((uintptr_t)qkv | (uintptr_t)q_rot | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;
    if (q16 && (!wide || T <= kBtMaxT)) return pi::fail(PI_E_ARG, "rope_kv_chunk: fp16 queries need rows of 16 bytes and more than 16 tokens");
    const int split = wide ? ((n_head + 2 * n_head_kv) * (hd / 8) + kBlock - 1) / kBlock : T >= 512 ? 1 : T >= 128 ? 4 : 16;
    const auto kernel = q16 ? rope_kv_chunk_wide_kernel<true> : wide ? rope_kv_chunk_wide_kernel<false> : rope_kv_chunk_kernel;
    hipLaunchKernelGGL(kernel, dim3(T, split), dim3(kBlock), sizeof(float2) * (hd / 2), st, qkv, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, q_rot,
                       (__half *)k_cache, (__half *)v_cache, qkv_stride, n_head * hd);
    return pi::check_launch("rope_kv_chunk");
}
bool attn_chunk_by_16(int hd, int n_kv_max) { return (hd == 64 || hd == 128) && chunk_mfma_lds(hd, n_kv_max) <= kChunkMfmaLds; }
}  // namespace pi

extern "C" {

int pi_k_rope_kv_store(const float * qkv, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                       const int32_t * pos, int n_ctx, float * q_rot, void * k_cache, void * v_cache, pi_stream_t stream) {
    if (!qkv || !pos || !q_rot || !k_cache || !v_cache) return pi::fail(PI_E_ARG, "pi_k_rope_kv_store: null pointer");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || hd <= 0 || hd % 2 || hd / 2 > 1024 || (mode != 0 && mode != 2))
        return pi::fail(PI_E_ARG, "pi_k_rope_kv_store: bad head geometry or mode");
    hipLaunchKernelGGL(rope_kv_store_kernel, dim3(n_head + 2 * n_head_kv), dim3(hd / 2), 0, (hipStream_t)stream,
                       qkv, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, q_rot, (__half *)k_cache, (__half *)v_cache, 0, 0);
    return pi::check_launch("pi_k_rope_kv_store");
}

int pi_k_attn_decode(const float * q_rot, const void * k_cache, const void * v_cache, int n_head, int n_head_kv,
                     int hd, int n_ctx, const int32_t * pos, float * out, pi_stream_t stream) {
    if (!q_rot || !k_cache || !v_cache || !pos || !out) return pi::fail(PI_E_ARG, "pi_k_attn_decode: null pointer");
    if (hd % 8 || kBlock % (hd / 8) || PI_WAVE % (hd / 8) || n_head % n_head_kv) return pi::fail(PI_E_ARG, "pi_k_attn_decode: head size must be 8 * (a divisor of 64)");
    const size_t sh = sizeof(float) * ((size_t)n_ctx + (size_t)(kBlock / (hd / 8)) * hd);
    if (sh > 60 * 1024) return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_decode: context too long for the single-pass kernel");
    hipLaunchKernelGGL(attn_decode_kernel, dim3(n_head), dim3(kBlock), sh, (hipStream_t)stream,
                       q_rot, (const __half *)k_cache, (const __half *)v_cache, n_head, n_head_kv, hd, n_ctx, pos, out, 0, 0, nullptr);
    return pi::check_launch("pi_k_attn_decode");
}

int pi_k_rope_table(void * table, int n_ctx, int hd, int mode, float theta_scale, float freq_scale, pi_stream_t stream) {
    if (!table || n_ctx <= 0 || hd <= 0 || hd % 2 || hd / 2 > 1024) return pi::fail(PI_E_ARG, "pi_k_rope_table: bad arguments");
    // A set-up call: the table is computed on the host with the C library's cosf / sinf -- the functions the CPU path itself calls
    // (ggml.c:11163-11325: theta = position, then *= theta_scale per pair) -- so rotated q and k start from bit-identical factors;
    // the device's own cosf / sinf may differ from them in the last place.
    const int half = hd / 2;
    std::vector<float> host((size_t)n_ctx * hd);
    for (int p = 0; p < n_ctx; ++p) {
        float theta = (mode & 2) ? (float)p * freq_scale : (float)p;             // rope_angle, one product per pair
        for (int i = 0; i < half; ++i) {
            const float th = freq_scale * theta;
            host[((size_t)p * half + i) * 2]     = cosf(th);
            host[((size_t)p * half + i) * 2 + 1] = sinf(th);
            theta *= theta_scale;
        }
    }
    PI_HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
    PI_HIP_TRY(hipMemcpy(table, host.data(), host.size() * sizeof(float), hipMemcpyHostToDevice));
    return PI_OK;
}

constexpr size_t kAttnLdsLimit = 60 * 1024;

int pi_k_attn_fused_supported(int hd, int n_ctx) {
    return attn_fused_geometry_ok(hd) && n_ctx > 0 && attn_fused_lds_bytes(hd, n_ctx) <= kAttnLdsLimit;
}

int pi_k_attn_decode_supported(int hd, int n_ctx) {
    return hd > 0 && hd % 8 == 0 && kBlock % (hd / 8) == 0 && PI_WAVE % (hd / 8) == 0 && n_ctx > 0 &&
           sizeof(float) * ((size_t)n_ctx + (size_t)(kBlock / (hd / 8)) * hd) <= kAttnLdsLimit;
}

}  // extern "C"

// the lanes of a cell are a constant for the two usual head sizes (their sums are then lane permutations)
#define PI_ATTN_LPP(...) do { if (hd == 128) { constexpr int LPP = 16; __VA_ARGS__; } else if (hd == 64) { constexpr int LPP = 8; __VA_ARGS__; } \
                              else { constexpr int LPP = 0; __VA_ARGS__; } } while (0)
// the parts and their merge
template <bool FROM_CACHE>
static int launch_attn_parts(const float * qkv, const float2 * rope_table, __half * k, __half * v, int n_tok, int n_head, int n_head_kv, int hd, int mode, int n_ctx, int n_parts, const int32_t * pos,
                             float * scratch, int qkv_stride, size_t cache_seq_stride, float * out, int out_stride, __half * out_f16, hipStream_t st, const char * name) {
    const int s_cap = (n_ctx + n_parts - 1) / n_parts + 1;
    const size_t lds = attn_part_lds(hd, s_cap);
    float * acc = scratch, * ml = scratch + (size_t)n_tok * n_head * n_parts * hd;
    PI_ATTN_LPP(hipLaunchKernelGGL((attn_part_kernel<FROM_CACHE, LPP>), dim3(n_head, n_parts, n_tok), dim3(kAttnPartBlock), lds, st, qkv, rope_table, k, v, n_head, n_head_kv, hd, mode, n_ctx, s_cap, pos, acc, ml,
                           qkv_stride, cache_seq_stride));
    hipLaunchKernelGGL(attn_merge_kernel, dim3(n_head, n_tok), dim3(hd), 0, st, acc, ml, n_parts, hd, out, out_stride, out_f16);
    return pi::check_launch(name);
}
namespace pi {
bool attn_out_small_supported(int n_head, int hd, int n_ctx) { return n_head <= kOutHeads && (hd == 64 || hd == 128) && pi_k_attn_fused_supported(hd, n_ctx); }
int attn_out_small(const DecodeAttn & a, const void * wo_f16, int d, float * parts, pi_stream_t stream) {
    if (!a.qkv || !a.rope_table || !a.k_cache || !a.v_cache || !a.pos || !wo_f16 || !parts || d <= 0 || ((uintptr_t)wo_f16 & 15)) return fail(PI_E_ARG, "attn_out_small: bad arguments");
    if (a.n_head <= 0 || a.n_head_kv <= 0 || a.n_head % a.n_head_kv || (a.mode != 0 && a.mode != 2) || !attn_out_small_supported(a.n_head, a.hd, a.n_ctx))
        return fail(PI_E_UNSUPPORTED, "attn_out_small: shape outside the kernel");
    const size_t sh = attn_fused_lds_bytes(a.hd, a.n_ctx);
    const auto kernel = a.hd == 128 ? attn_out_small_kernel<16> : attn_out_small_kernel<8>;
    hipLaunchKernelGGL(kernel, dim3(a.n_head), dim3(kAttnBlock), sh, (hipStream_t)stream, a.qkv, (const float2 *)a.rope_table, (__half *)a.k_cache, (__half *)a.v_cache, a.n_head, a.n_head_kv, a.hd, a.mode,
                       a.n_ctx, a.pos, (const __half *)wo_f16, d, parts);
    return check_launch("attn_out_small");
}
int attn_fused(const float * qkv, const void * rope_table, void * k_cache, void * v_cache, int n_head, int n_head_kv, int hd, int mode,
               int n_ctx, const int32_t * pos, float * out, const Ahead & ahead, pi_stream_t stream) {
    if (!qkv || !rope_table || !k_cache || !v_cache || !pos || !out) return pi::fail(PI_E_ARG, "pi_k_attn_fused: null pointer");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || !attn_fused_geometry_ok(hd) || (mode != 0 && mode != 2))
        return pi::fail(PI_E_ARG, "pi_k_attn_fused: head size must be 8 * (a divisor of 64), at most 128; mode 0 or 2");
    const size_t sh = attn_fused_lds_bytes(hd, n_ctx);
    if (sh > kAttnLdsLimit) return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_fused: context too long for the single-pass kernel");
    PI_ATTN_LPP(hipLaunchKernelGGL((attn_fused_kernel<kAttnBlock, LPP>), dim3(n_head + ahead.blocks), dim3(kAttnBlock), sh, (hipStream_t)stream, qkv, (const float2 *)rope_table,
                       (__half *)k_cache, (__half *)v_cache, n_head, n_head_kv, hd, mode, n_ctx, pos, out, 0, (size_t)0, 0, nullptr, 0, nullptr, nullptr, nullptr, ahead));
    return pi::check_launch("pi_k_attn_fused");
}
}  // namespace pi
extern "C" {
int pi_k_attn_fused(const float * qkv, const void * rope_table, void * k_cache, void * v_cache, int n_head, int n_head_kv, int hd, int mode,
                    int n_ctx, const int32_t * pos, float * out, pi_stream_t stream) {
    return pi::attn_fused(qkv, rope_table, k_cache, v_cache, n_head, n_head_kv, hd, mode, n_ctx, pos, out, pi::Ahead{}, stream);
}

// ---- attention with the cells of a head split over n_parts workgroups --------------------------------------------
static bool attn_part_geometry_ok(int hd) {
    return hd > 0 && hd % 8 == 0 && kAttnPartBlock % (hd / 8) == 0 && PI_WAVE % (hd / 8) == 0 && hd / 2 + hd <= kAttnPartBlock && hd <= 1024;
}
int pi_k_attn_split_supported(int hd, int n_ctx, int n_parts) {
    return attn_part_geometry_ok(hd) && n_ctx > 0 && n_parts >= 1 && n_parts <= 64 && attn_part_lds(hd, (n_ctx + n_parts - 1) / n_parts + 1) <= kAttnLdsLimit;
}
size_t pi_k_attn_split_scratch_floats(int n_seq, int n_head, int hd, int n_parts) { return (size_t)n_seq * n_head * n_parts * ((size_t)hd + 2); }

int pi_k_attn_split(const float * qkv, int qkv_stride, const void * rope_table, void * k_cache, void * v_cache, size_t cache_seq_stride,
                    int n_seq, int n_head, int n_head_kv, int hd, int mode, int n_ctx, int n_parts, const int32_t * pos, float * scratch,
                    float * out, int out_stride, void * out_f16, pi_stream_t stream) {
    if (!qkv || !rope_table || !k_cache || !v_cache || !pos || !out || !scratch || n_seq <= 0) return pi::fail(PI_E_ARG, "pi_k_attn_split: bad arguments");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || (mode != 0 && mode != 2) || !pi_k_attn_split_supported(hd, n_ctx, n_parts))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_split: head size, context per part or part count outside the kernel (pi_k_attn_split_supported)");
    return launch_attn_parts<false>(qkv, (const float2 *)rope_table, (__half *)k_cache, (__half *)v_cache, n_seq, n_head, n_head_kv, hd, mode, n_ctx, n_parts, pos, scratch, qkv_stride,
                                    cache_seq_stride, out, out_stride, (__half *)out_f16, (hipStream_t)stream, "pi_k_attn_split");
}

int pi_k_attn_split_cached(const float * q_rot, const void * k_cache, const void * v_cache, int n_tok, int n_head, int n_head_kv, int hd,
                           int n_ctx, int n_parts, const int32_t * pos, float * scratch, float * out, pi_stream_t stream) {
    if (!q_rot || !k_cache || !v_cache || !pos || !out || !scratch || n_tok <= 0 || n_tok > 65535) return pi::fail(PI_E_ARG, "pi_k_attn_split_cached: bad arguments");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || !pi_k_attn_split_supported(hd, n_ctx, n_parts))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_split_cached: head size, context per part or part count outside the kernel (pi_k_attn_split_supported)");
    return launch_attn_parts<true>(q_rot, nullptr, (__half *)const_cast<void *>(k_cache), (__half *)const_cast<void *>(v_cache), n_tok, n_head, n_head_kv, hd, 0, n_ctx, n_parts, pos, scratch,
                                   n_head * hd, 0, out, n_head * hd, nullptr, (hipStream_t)stream, "pi_k_attn_split_cached");
}

static int attn_fused_batch(const float * qkv, int qkv_stride, const void * rope_table, void * k_cache, void * v_cache, size_t cache_seq_stride,
                            int n_seq, int n_head, int n_head_kv, int hd, int mode, int n_ctx, const int32_t * pos, float * out, int out_stride,
                            void * out_f16, pi_stream_t stream, int out16_ol, void * q8_q = nullptr, float * q8_d = nullptr, int32_t * q8_s = nullptr) {
    if (q8_q && (hd % 32 || !q8_d || !q8_s)) return pi::fail(PI_E_ARG, "pi_k_attn_fused_batch_q8: head size % 32 == 0 and all three outputs required");
    if (!qkv || !rope_table || !k_cache || !v_cache || !pos || !out || n_seq <= 0 || n_seq > kBtMaxT) return pi::fail(PI_E_ARG, "pi_k_attn_fused_batch: bad arguments");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || !attn_fused_geometry_ok(hd) || (mode != 0 && mode != 2))
        return pi::fail(PI_E_ARG, "pi_k_attn_fused_batch: head size must be 8 * (a divisor of 64), at most 128; mode 0 or 2");
    const size_t sh = attn_fused_lds_bytes(hd, n_ctx);
    if (sh > kAttnLdsLimit) return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_fused_batch: context too long for the single-pass kernel");
    const int n_cu = pi::compute_units();
    if (n_cu > 0 && n_seq * n_head > 2 * n_cu)
        PI_ATTN_LPP(hipLaunchKernelGGL((attn_fused_kernel<kAttnBlock / 2, LPP>), dim3(n_head, n_seq), dim3(kAttnBlock / 2), attn_fused_lds_bytes(hd, n_ctx, kAttnBlock / 2), (hipStream_t)stream, qkv, (const float2 *)rope_table,
                           (__half *)k_cache, (__half *)v_cache, n_head, n_head_kv, hd, mode, n_ctx, pos, out, qkv_stride, cache_seq_stride, out_stride, (__half *)out_f16, out16_ol, (int8_t *)q8_q, q8_d, q8_s, Ahead{}));
    else
        PI_ATTN_LPP(hipLaunchKernelGGL((attn_fused_kernel<kAttnBlock, LPP>), dim3(n_head, n_seq), dim3(kAttnBlock), sh, (hipStream_t)stream, qkv, (const float2 *)rope_table,
                           (__half *)k_cache, (__half *)v_cache, n_head, n_head_kv, hd, mode, n_ctx, pos, out, qkv_stride, cache_seq_stride, out_stride, (__half *)out_f16, out16_ol, (int8_t *)q8_q, q8_d, q8_s, Ahead{}));
    return pi::check_launch("pi_k_attn_fused_batch");
}

int pi_k_attn_fused_batch(const float * qkv, int qkv_stride, const void * rope_table, void * k_cache, void * v_cache, size_t cache_seq_stride,
                          int n_seq, int n_head, int n_head_kv, int hd, int mode, int n_ctx, const int32_t * pos, float * out, int out_stride,
                          void * out_f16, pi_stream_t stream) {
    return attn_fused_batch(qkv, qkv_stride, rope_table, k_cache, v_cache, cache_seq_stride, n_seq, n_head, n_head_kv, hd, mode, n_ctx, pos, out, out_stride, out_f16, stream, 0);
}

int pi_k_attn_fused_batch_q8(const float * qkv, int qkv_stride, const void * rope_table, void * k_cache, void * v_cache, size_t cache_seq_stride,
                             int n_seq, int n_head, int n_head_kv, int hd, int mode, int n_ctx, const int32_t * pos, float * out, int out_stride,
                             void * q8_quants, float * q8_scales, int32_t * q8_sums, pi_stream_t stream) {
    if (!q8_quants) return pi::fail(PI_E_ARG, "pi_k_attn_fused_batch_q8: null pointer");
    return attn_fused_batch(qkv, qkv_stride, rope_table, k_cache, v_cache, cache_seq_stride, n_seq, n_head, n_head_kv, hd, mode, n_ctx, pos, out, out_stride, nullptr, stream, 0,
                            q8_quants, q8_scales, q8_sums);
}

int pi_k_attn_fused_batch_ol(const float * qkv, int qkv_stride, const void * rope_table, void * k_cache, void * v_cache, size_t cache_seq_stride,
                             int n_seq, int n_head, int n_head_kv, int hd, int mode, int n_ctx, const int32_t * pos, float * out, int out_stride,
                             void * out_ol, pi_stream_t stream) {
    return attn_fused_batch(qkv, qkv_stride, rope_table, k_cache, v_cache, cache_seq_stride, n_seq, n_head, n_head_kv, hd, mode, n_ctx, pos, out, out_stride, out_ol, stream, 1);
}

static int attn_chunk(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                    const int32_t * pos, int n_ctx, int n_kv_max, float * q_rot, void * k_cache, void * v_cache, float * out, int out_stride, void * out_f16,
                      int q8, pi_stream_t stream) {
    if (!qkv || !pos || !q_rot || !k_cache || !v_cache || (q8 ? !out_f16 : !out) || T <= 0 || T > kChunkMaxT) return pi::fail(PI_E_ARG, "pi_k_attn_chunk: bad arguments");
    if (n_kv_max <= 0 || n_kv_max > n_ctx) n_kv_max = n_ctx;                  // cells the furthest token of the chunk attends: what the scores in LDS are sized for
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || hd <= 0 || hd % 8 || hd / 2 > 1024 || kBlock % (hd / 8) || PI_WAVE % (hd / 8) || (mode != 0 && mode != 2))
        return pi::fail(PI_E_ARG, "pi_k_attn_chunk: bad head geometry or mode");
    hipStream_t st = (hipStream_t)stream;
    // all K/V rows of the chunk are in the cache before any token of the chunk attends
    const int rc = pi::rope_kv_chunk(qkv, qkv_stride, T, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, q_rot, k_cache, v_cache, st);
    if (rc != PI_OK) return rc;
    // 16 tokens per workgroup on the matrix cores where the head size and the context fit (scores of 16 tokens in LDS)
    const char * own = getenv("PI_ATTN_CHUNK");
    const bool scalar = own && !strcmp(own, "scalar");
    const int s_stride = ((n_kv_max + 31) & ~31) + 4;
    const size_t sh_mfma = chunk_mfma_lds(hd, n_kv_max);
    if ((hd == 128 || hd == 64) && T > 1 && sh_mfma <= kChunkMfmaLds && !scalar) {
        static bool raised[2] = {false, false};
        if (!raised[hd == 64]) {
            if (hd == 128) PI_HIP_TRY(hipFuncSetAttribute((const void *)attn_chunk_mfma_kernel<128>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kChunkMfmaLds));
            else           PI_HIP_TRY(hipFuncSetAttribute((const void *)attn_chunk_mfma_kernel<64>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kChunkMfmaLds));
            raised[hd == 64] = true;
        }
        const dim3 grid(n_head, (T + 15) / 16);
        if (hd == 128) hipLaunchKernelGGL(attn_chunk_mfma_kernel<128>, grid, dim3(kBlock), sh_mfma, st, q_rot, (const __half *)k_cache, (const __half *)v_cache,
                                          n_head, n_head_kv, n_ctx, pos, T, out, n_head * hd, out_stride, (__half *)out_f16, s_stride, q8);
        else           hipLaunchKernelGGL(attn_chunk_mfma_kernel<64>, grid, dim3(kBlock), sh_mfma, st, q_rot, (const __half *)k_cache, (const __half *)v_cache,
                                          n_head, n_head_kv, n_ctx, pos, T, out, n_head * hd, out_stride, (__half *)out_f16, s_stride, q8);
        return pi::check_launch("pi_k_attn_chunk");
    }
    if (q8) return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_chunk_q8: head sizes 64 and 128, several tokens, cells whose scores fit");
    const size_t sh = sizeof(float) * ((size_t)n_ctx + (size_t)(kBlock / (hd / 8)) * hd);
    if (sh > 60 * 1024) return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_chunk: context too long for the single-pass kernel (pi_k_attn_chunk_supported)");
    hipLaunchKernelGGL(attn_decode_kernel, dim3(n_head, T), dim3(kBlock), sh, st,
                       q_rot, (const __half *)k_cache, (const __half *)v_cache, n_head, n_head_kv, hd, n_ctx, pos, out, n_head * hd, out_stride, (__half *)out_f16);
    return pi::check_launch("pi_k_attn_chunk");
}

int pi_k_attn_chunk(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                    const int32_t * pos, int n_ctx, int n_kv_max, float * q_rot, void * k_cache, void * v_cache, float * out, int out_stride, void * out_f16,
                    pi_stream_t stream) {
    return attn_chunk(qkv, qkv_stride, T, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, n_kv_max, q_rot, k_cache, v_cache, out, out_stride, out_f16, 0, stream);
}

int pi_k_attn_chunk_q8(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                       const int32_t * pos, int n_ctx, int n_kv_max, float * q_rot, void * k_cache, void * v_cache, int cols, void * out_f16, int ol,
                       pi_stream_t stream) {
    return attn_chunk(qkv, qkv_stride, T, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, n_kv_max, q_rot, k_cache, v_cache, nullptr, cols, out_f16, ol ? 2 : 1, stream);
}

// where attn_chunk_rows_kernel is the faster one: fewer than 32 tokens against many cells are better off with attn_chunk_mfma_kernel, whose waves
// split the cells (32 heads of 128, 17 tokens: 59 against 49 us at 1817 cells, 17.5 and 17.7 at 317; 48 tokens, 1848 cells: 91 and 102)
int pi_k_attn_chunk_rows_supported(int hd, int T, int n_kv_max) {
    return (hd == 64 || hd == 128) && T > kBtMaxT && n_kv_max > 0 && (T >= 32 || n_kv_max <= 512 || chunk_mfma_lds(hd, n_kv_max) > kChunkMfmaLds);
}

int pi_k_attn_chunk_rows(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                         const int32_t * pos, int n_ctx, int n_kv_max, float * q_rot, void * k_cache, void * v_cache, float * out, int out_stride, void * out_f16,
                         pi_stream_t stream) {
    if (!qkv || !pos || !q_rot || !k_cache || !v_cache || !out || T <= 0 || n_ctx <= 0) return pi::fail(PI_E_ARG, "pi_k_attn_chunk_rows: bad arguments");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || (hd != 64 && hd != 128) || (mode != 0 && mode != 2)) return pi::fail(PI_E_ARG, "pi_k_attn_chunk_rows: bad head geometry or mode");
    if (out_stride % 4 || (((uintptr_t)q_rot | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) || ((uintptr_t)out_f16 & 7))
        return pi::fail(PI_E_ARG, "pi_k_attn_chunk_rows: rows of whole quads, buffers on 16 bytes (out_f16: 8)");
    if (n_kv_max <= 0 || n_kv_max > n_ctx) n_kv_max = n_ctx;
    hipStream_t st = (hipStream_t)stream;
    const int rc = pi::rope_kv_chunk(qkv, qkv_stride, T, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, q_rot, k_cache, v_cache, st);
    if (rc != PI_OK) return rc;
    // 128 tokens a workgroup where that still leaves two for every compute unit
    const bool two = (long long)n_head * ((T + 127) / 128) >= 2 * pi::compute_units();
    // pi_k_attn_chunk's rounding points where it covers the cache; no more than pi_k_attn_chunk_long's beyond
    const bool whole = !pi_k_attn_chunk_supported(hd, n_ctx, n_kv_max);
#define PI_ROWS(HD, U, W) launch_chunk_rows<HD, U, W>(q_rot, k_cache, v_cache, n_head, n_head_kv, n_ctx, pos, T, n_kv_max, out, out_stride, out_f16, st)
#define PI_ROWS_U(HD, U) (whole ? PI_ROWS(HD, U, true) : PI_ROWS(HD, U, false))
    return hd == 128 ? (two ? PI_ROWS_U(128, 2) : PI_ROWS_U(128, 1)) : (two ? PI_ROWS_U(64, 2) : PI_ROWS_U(64, 1));
#undef PI_ROWS_U
#undef PI_ROWS
}

int pi_k_attn_chunk_once(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                         const int32_t * pos, int n_ctx, int n_kv_max, void * q_f16, void * k_cache, void * v_cache, float * out, int out_stride, void * out_f16,
                         pi_stream_t stream) {
    if (!qkv || !pos || !q_f16 || !k_cache || !v_cache || (!out && !out_f16) || T <= kBtMaxT || n_ctx <= 0) return pi::fail(PI_E_ARG, "pi_k_attn_chunk_once: bad arguments");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || (hd != 64 && hd != 128) || (mode != 0 && mode != 2)) return pi::fail(PI_E_ARG, "pi_k_attn_chunk_once: bad head geometry or mode");
    if (qkv_stride % 4 || out_stride % 4 || (((uintptr_t)qkv | (uintptr_t)q_f16 | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) || ((uintptr_t)out_f16 & 7))
        return pi::fail(PI_E_ARG, "pi_k_attn_chunk_once: rows of whole quads, buffers on 16 bytes (out_f16: 8)");
    if (n_kv_max <= 0 || n_kv_max > n_ctx) n_kv_max = n_ctx;
    hipStream_t st = (hipStream_t)stream;
    const int rc = pi::rope_kv_chunk(qkv, qkv_stride, T, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, (float *)q_f16, k_cache, v_cache, st, true);
    if (rc != PI_OK) return rc;
    const bool two = (long long)n_head * ((T + 127) / 128) >= 2 * pi::compute_units();
#define PI_ONCE(HD, U) launch_chunk_once<HD, U>(q_f16, k_cache, v_cache, n_head, n_head_kv, n_ctx, pos, T, n_kv_max, out, out_stride, out_f16, st)
    return hd == 128 ? (two ? PI_ONCE(128, 2) : PI_ONCE(128, 1)) : (two ? PI_ONCE(64, 2) : PI_ONCE(64, 1));
#undef PI_ONCE
}

int pi_k_attn_chunk_supported(int hd, int n_ctx, int n_kv_max) {
    if (hd <= 0 || hd % 8 || kBlock % (hd / 8) || PI_WAVE % (hd / 8) || n_ctx <= 0) return 0;
    if (n_kv_max <= 0 || n_kv_max > n_ctx) n_kv_max = n_ctx;
    if (pi::attn_chunk_by_16(hd, n_kv_max)) return 1;
    return sizeof(float) * ((size_t)n_ctx + (size_t)(kBlock / (hd / 8)) * hd) <= 60 * 1024;
}

// pi_k_attn_chunk for contexts beyond its kernels: RoPE + KV store of the chunk, then every token's cells split over n_parts workgroups
int pi_k_attn_chunk_long(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale,
                         const int32_t * pos, int n_ctx, int n_parts, float * scratch, float * q_rot, void * k_cache, void * v_cache,
                         float * out, void * out_f16, pi_stream_t stream) {
    if (!qkv || !pos || !q_rot || !k_cache || !v_cache || !out || !scratch || T <= 0 || T > kChunkMaxT) return pi::fail(PI_E_ARG, "pi_k_attn_chunk_long: bad arguments");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || (mode != 0 && mode != 2) || hd % 2 || hd / 2 > 1024 || !pi_k_attn_split_supported(hd, n_ctx, n_parts))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_chunk_long: head size, context per part or part count outside the kernel (pi_k_attn_split_supported)");
    hipStream_t st = (hipStream_t)stream;
    const int rc = pi::rope_kv_chunk(qkv, qkv_stride, T, n_head, n_head_kv, hd, mode, theta_scale, freq_scale, pos, n_ctx, q_rot, k_cache, v_cache, st);
    if (rc != PI_OK) return rc;
    return launch_attn_parts<true>(q_rot, nullptr, (__half *)k_cache, (__half *)v_cache, T, n_head, n_head_kv, hd, 0, n_ctx, n_parts, pos, scratch, n_head * hd, 0, out, n_head * hd,
                                   (__half *)out_f16, st, "pi_k_attn_chunk_long");
}

static size_t attn_ggml_lds(int hd, int n_kv, int T) {
    return sizeof(float) * (size_t)((n_kv + 7) & ~7) + 2 * (size_t)hd * (1 + 2 * (size_t)T) + sizeof(float) * kBlock;
}
int pi_k_attn_ggml_supported(int hd, int n_ctx, int n_kv) {
    return hd > 0 && hd % 8 == 0 && hd <= kBlock && kBlock % hd == 0 && PI_WAVE % (hd / 8) == 0 && n_kv > 0 && n_ctx % 8 == 0 && n_kv <= n_ctx &&
           attn_ggml_lds(hd, n_kv, kBtMaxT) <= 60 * 1024;
}

int pi_k_attn_ggml(const float * q, const float * k, const float * v, const int32_t * pos, int mode, float theta_scale, float freq_scale, float mscale,
                   void * k_cache, void * v_cache, int n_head, int n_head_kv, int hd, int n_ctx, int n_kv, int cell,
                   const float * kq_scale, const float * kq_mask, float * out, pi_stream_t stream) {
    if (!q || !k || !v || !pos || !k_cache || !v_cache || !kq_scale || !kq_mask || !out) return pi::fail(PI_E_ARG, "pi_k_attn_ggml: null pointer");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || (mode != 0 && mode != 2) || cell < 0 || cell >= n_kv || !pi_k_attn_ggml_supported(hd, n_ctx, n_kv))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_ggml: head geometry, cell or context outside the kernel (pi_k_attn_ggml_supported)");
    if ((((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) != 0) return pi::fail(PI_E_ARG, "pi_k_attn_ggml: the caches must be 16-byte aligned");
    hipLaunchKernelGGL(attn_ggml_kernel, dim3(n_head, 1), dim3(kBlock), attn_ggml_lds(hd, n_kv, 1), (hipStream_t)stream, q, k, v, 0, pos, mode, theta_scale, freq_scale, mscale,
                       (__half *)k_cache, (__half *)v_cache, n_head, n_head_kv, hd, n_ctx, n_kv, 1, cell, kq_scale, kq_mask, 0, out, 0);
    return pi::check_launch("pi_k_attn_ggml");
}

int pi_k_attn_ggml_step(const float * qkv, int qkv_stride, const int32_t * pos, int mode, float theta_scale, float freq_scale, float mscale,
                        void * k_cache, void * v_cache, int n_head, int n_head_kv, int hd, int n_ctx, int n_kv, int T, int cell0,
                        const float * kq_scale, const float * kq_mask, int mask_stride, float * out, int out_stride, pi_stream_t stream) {
    if (!qkv || !pos || !k_cache || !v_cache || !kq_scale || !kq_mask || !out) return pi::fail(PI_E_ARG, "pi_k_attn_ggml_step: null pointer");
    if (n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv || (mode != 0 && mode != 2) || T < 1 || T > kBtMaxT || cell0 < 0 || cell0 + T > n_kv ||
        qkv_stride < (n_head + 2 * n_head_kv) * hd || mask_stride < n_kv || out_stride < n_head * hd || !pi_k_attn_ggml_supported(hd, n_ctx, n_kv))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_attn_ggml_step: head geometry, cells, strides or context outside the kernel (pi_k_attn_ggml_supported)");
    if ((((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) != 0) return pi::fail(PI_E_ARG, "pi_k_attn_ggml_step: the caches must be 16-byte aligned");
    hipLaunchKernelGGL(attn_ggml_kernel, dim3(n_head, T), dim3(kBlock), attn_ggml_lds(hd, n_kv, T), (hipStream_t)stream, qkv, qkv + (size_t)n_head * hd,
                       qkv + (size_t)(n_head + n_head_kv) * hd, qkv_stride, pos, mode, theta_scale, freq_scale, mscale, (__half *)k_cache, (__half *)v_cache,
                       n_head, n_head_kv, hd, n_ctx, n_kv, T, cell0, kq_scale, kq_mask, mask_stride, out, out_stride);
    return pi::check_launch("pi_k_attn_ggml_step");
}

int pi_k_k_shift(void * k_cache, int rows, int n_ctx, int hd, int mode, float theta_scale, float freq_scale, const int32_t * delta, int n_cells, pi_stream_t stream) {
    if (!k_cache || !delta || rows <= 0 || n_ctx <= 0 || hd <= 0 || hd % 2 || hd / 2 > 1024 || n_cells < 0 || n_cells > n_ctx || (mode != 0 && mode != 2))
        return pi::fail(PI_E_ARG, "pi_k_k_shift: bad arguments");
    if (n_cells == 0) return PI_OK;
    hipLaunchKernelGGL(k_shift_kernel, dim3(n_cells, rows), dim3(hd / 2), 0, (hipStream_t)stream, (__half *)k_cache, n_ctx, hd, mode, theta_scale, freq_scale, delta);
    return pi::check_launch("pi_k_k_shift");
}

int pi_k_k_shift_cells(void * k_cache, int n_layer, int n_cells, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale, const int32_t * delta,
                       pi_stream_t stream) {
    if (!k_cache || !delta || n_layer <= 0 || n_cells <= 0 || n_head_kv <= 0 || hd <= 0 || hd % 2 || hd / 2 > 1024 || (mode != 0 && mode != 2))
        return pi::fail(PI_E_ARG, "pi_k_k_shift_cells: bad arguments");
    hipLaunchKernelGGL(k_shift_cells_kernel, dim3(n_cells, n_layer * n_head_kv), dim3(hd / 2), 0, (hipStream_t)stream, (__half *)k_cache, n_cells, n_head_kv, hd, mode,
                       theta_scale, freq_scale, delta);
    return pi::check_launch("pi_k_k_shift_cells");
}

int pi_k_kv_compact(void * cache, void * stage, int rows, int n_ctx, int hd, const int32_t * map, int n_new, pi_stream_t stream) {
    if (!cache || !stage || !map || rows <= 0 || n_ctx <= 0 || hd <= 0 || hd % 8 || hd / 8 > 1024 || n_new < 0 || n_new > n_ctx)
        return pi::fail(PI_E_ARG, "pi_k_kv_compact: bad arguments");
    if (n_new == 0) return PI_OK;
    hipLaunchKernelGGL(kv_gather_kernel, dim3(n_new, rows), dim3(hd / 8), 0, (hipStream_t)stream, (const __half *)cache, (__half *)stage, map, n_new, n_ctx, hd);
    hipLaunchKernelGGL(kv_place_kernel, dim3(n_new, rows), dim3(hd / 8), 0, (hipStream_t)stream, (__half *)cache, (const __half *)stage, n_new, n_ctx, hd);
    return pi::check_launch("pi_k_kv_compact");
}

}  // extern "C"
