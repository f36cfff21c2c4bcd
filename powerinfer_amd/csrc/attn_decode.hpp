// Attention of decoded tokens: the device code of its launches, which a launch of the sparse FFN takes along.
#pragma once
#include "kernels_common.hpp"

namespace {

// ---------------------------------------------------------------------------------------------------
// RoPE + KV store + decode attention in one launch, one workgroup per query head.  The workgroup rotates its
// own q head and the k head of its group (cos/sin from the table), rounds k and v to fp16 as the cache does,
// and attends over cells [0, pos) from the cache plus the new cell from LDS, so it never reads what this
// launch writes; the first query head of each group stores k and v.
// ---------------------------------------------------------------------------------------------------
constexpr int kAttnBlock = 1024;        // 16 waves per head: 64 (hd 128) or 128 (hd 64) cache cells per pass
constexpr int kAttnPre = 4;             // passes whose K and V rows are requested before the prologue
constexpr int kAttnBatch = 4;           // passes behind those whose rows are requested together
// BLOCK threads per head: kAttnBlock for a single sequence and for steps whose workgroups all fit on the chip at once (two of 1024
// threads per compute unit); half of that where they do not (16 sequences x 40 heads are 640 workgroups against 512 places: a
// quarter of the units ran a second round, 48 us at 530 cells; with 512 threads four fit a unit and all 640 run together).
// LPP: hd / 8, the lanes of a cell, where it is 16 or 8 (0: any)
template <int BLOCK, int LPP>
__device__ __forceinline__ void attn_fused_head(const float * __restrict__ qkv, const float2 * __restrict__ rope_table,
                                                            __half * __restrict__ k_cache, __half * __restrict__ v_cache,
                                                            int n_head, int n_head_kv, int hd, int mode, int n_ctx,
                                                            const int32_t * __restrict__ pos_p, float * __restrict__ out,
                                                            int qkv_stride, size_t cache_seq_stride, int out_stride, __half * __restrict__ out16, int out16_ol,
                                                            int8_t * __restrict__ q8_q, float * __restrict__ q8_d, int * __restrict__ q8_s,
                                                const int h, const int y, __half * out_lds = nullptr) {
    // out_lds: instead of out, this head's values in fp16
    // q8_q != nullptr: the output also as the Q8_0 blocks an integer mat-mul of a Q4_0 matrix multiplies with (the blocks, scales and
    // -8 * sums pi_k_norm_q8_blocks makes of the same values: a head's hd outputs are whole blocks of 32, one per half-wave)
    // y: sequence of a batched step (its own token, position and cache); 0 for single-sequence decoding
    // out16_ol != 0: the fp16 copy in the operand layout of the 16-token mat-muls (pi_ol_index) instead of [sequence][out_stride]
    qkv += (size_t)y * qkv_stride;
    k_cache += (size_t)y * cache_seq_stride;
    v_cache += (size_t)y * cache_seq_stride;
    if (!out_lds) out += (size_t)y * out_stride;
    if (out16 && !out16_ol) out16 += (size_t)y * out_stride;      // optional fp16 copy: the input of the next mat-mul of a batched step
    pos_p += y;
    extern __shared__ __align__(16) unsigned char smem[];
    float * s    = reinterpret_cast<float *>(smem);               // [n_ctx] scores, then probabilities
    float * part = s + n_ctx;                                     // [groups][hd]
    float * qs   = part + (BLOCK / (hd / 8)) * hd;                    // [hd] rotated q, rounded to fp16
    float * kcur = qs + hd;                                       // [hd] rotated k of this position, rounded to fp16
    float * vcur = kcur + hd;                                     // [hd]
    __shared__ double red[16];
    __shared__ float redf[16];
    const int grp_sz = n_head / n_head_kv, kvh = h / grp_sz;
    const int tid = threadIdx.x;
    const int pos = *pos_p, n_kv = pos + 1;
    const float * qsrc = qkv + (size_t)h * hd;
    const float * ksrc = qkv + (size_t)(n_head + kvh) * hd;
    const float * vsrc = qkv + (size_t)(n_head + n_head_kv + kvh) * hd;
    __half * kdst = k_cache + ((size_t)kvh * n_ctx + pos) * hd;
    __half * vdst = v_cache + ((size_t)kvh * n_ctx + pos) * hd;
    const bool leader = (h % grp_sz) == 0;
    // the cache cells of the first kAttnPre passes do not depend on anything computed here: their K and V rows are requested
    // now and travel during the rotation, the scores and the softmax (one memory round trip instead of three in a row)
    const int lpp = LPP ? LPP : hd / 8;
    const int sub = tid % lpp, grp = tid / lpp, ngrp = BLOCK / lpp;
    const __half * kb = k_cache + (size_t)kvh * n_ctx * hd;
    const __half * vb = v_cache + (size_t)kvh * n_ctx * hd;
    pi_u32x4 kpre[kAttnPre], vpre[kAttnPre];
#pragma unroll
    for (int i = 0; i < kAttnPre; ++i) {
        const int c = i * ngrp + grp;
        if (c < pos) { kpre[i] = pi_ld16(kb + (size_t)c * hd + sub * 8); vpre[i] = pi_ld16(vb + (size_t)c * hd + sub * 8); }
    }
    if (tid < hd / 2) {
        const float2 cs = rope_table[(size_t)pos * (hd / 2) + tid];
        const int i0 = (mode & 2) ? tid : 2 * tid;
        const int i1 = (mode & 2) ? tid + hd / 2 : 2 * tid + 1;
        const float q0 = qsrc[i0], q1 = qsrc[i1], k0 = ksrc[i0], k1 = ksrc[i1];
        qs[i0] = pi_round_f16(__fsub_rn(__fmul_rn(q0, cs.x), __fmul_rn(q1, cs.y)));
        qs[i1] = pi_round_f16(__fadd_rn(__fmul_rn(q0, cs.y), __fmul_rn(q1, cs.x)));
        const __half ka = __float2half_rn(__fsub_rn(__fmul_rn(k0, cs.x), __fmul_rn(k1, cs.y)));
        const __half kb = __float2half_rn(__fadd_rn(__fmul_rn(k0, cs.y), __fmul_rn(k1, cs.x)));
        kcur[i0] = __half2float(ka); kcur[i1] = __half2float(kb);
        if (leader) { kdst[i0] = ka; kdst[i1] = kb; }
    } else if (tid < hd / 2 + hd) {
        const int e = tid - hd / 2;
        const __half v = __float2half_rn(vsrc[e]);
        vcur[e] = __half2float(v);
        if (leader) vdst[e] = v;
    }
    __syncthreads();

    const float scale = pi_inv_sqrt((float)hd);
    float qf[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) qf[i] = qs[sub * 8 + i];
#pragma unroll
    for (int i = 0; i < kAttnPre; ++i) {                            // (a row past the last is whatever the registers hold, and not used)
        if (i * ngrp < pos) {
            const int c = i * ngrp + grp;
            const float d = pi_group_sum<LPP>(pi_dot8(kpre[i], qf, 0.0f), lpp);
            if (c < pos && sub == 0) s[c] = __fmul_rn(d, scale);
        }
    }
    if (grp == pos % ngrp) {                                        // the new cell
        float d = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) d = fmaf(kcur[sub * 8 + k], qf[k], d);
        d = pi_group_sum<LPP>(d, lpp);
        if (sub == 0) s[pos] = __fmul_rn(d, scale);
    }
    // the passes behind the prefetched ones, kAttnBatch at a time: their rows are requested together and cost one trip to memory
    // instead of one each (the same dots in the same order)
    for (int c0 = kAttnPre * ngrp; c0 < pos; c0 += kAttnBatch * ngrp) {
        pi_u32x4 kk[kAttnBatch];
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            const int c = c0 + u * ngrp + grp;
            if (c < pos) kk[u] = pi_ld16(kb + (size_t)c * hd + sub * 8);
        }
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            if (c0 + u * ngrp < pos) {
                const int c = c0 + u * ngrp + grp;
                const float d = pi_group_sum<LPP>(pi_dot8(kk[u], qf, 0.0f), lpp);
                if (c < pos && sub == 0) s[c] = __fmul_rn(d, scale);
            }
        }
    }
    __syncthreads();

    float mx = -INFINITY;
    for (int c = tid; c < n_kv; c += BLOCK) mx = fmaxf(mx, s[c]);
    mx = block_max_f32(mx, redf);
    double sum = 0.0;
    for (int c = tid; c < n_kv; c += BLOCK) {
        const float e = pi_round_f16(expf(pi_round_f16(__fsub_rn(s[c], mx))));
        s[c] = e;
        sum += (double)e;
    }
    sum = block_sum_f64(sum, red);
    const float inv = (float)(1.0 / sum);

    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < kAttnPre; ++i) {
        const int c = i * ngrp + grp;
        if (c < n_kv) {
            const float p = pi_round_f16(__fmul_rn(s[c], inv));
            float vf[8];
            if (c < pos) pi_unpack8(vpre[i], vf);
            else {
#pragma unroll
                for (int k = 0; k < 8; ++k) vf[k] = vcur[sub * 8 + k];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = fmaf(vf[k], p, acc[k]);
        }
    }
    for (int c0 = kAttnPre * ngrp; c0 < n_kv; c0 += kAttnBatch * ngrp) {
        pi_u32x4 vv[kAttnBatch];
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            const int c = c0 + u * ngrp + grp;
            if (c < pos) vv[u] = pi_ld16(vb + (size_t)c * hd + sub * 8);
        }
#pragma unroll
        for (int u = 0; u < kAttnBatch; ++u) {
            const int c = c0 + u * ngrp + grp;
            if (c < n_kv) {
                const float p = pi_round_f16(__fmul_rn(s[c], inv));
                float vf[8];
                if (c < pos) pi_unpack8(vv[u], vf);
                else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) vf[i] = vcur[sub * 8 + i];
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[i] = fmaf(vf[i], p, acc[i]);
            }
        }
    }
    // (fewer cells than groups: the groups behind hold zeros, of which one is added for all)
    const int n_grp = min(ngrp, (n_kv + 7) & ~7);
    if (grp < n_grp) {
#pragma unroll
        for (int i = 0; i < 8; ++i) part[grp * hd + sub * 8 + i] = acc[i];
    }
    __syncthreads();
    for (int e = tid; e < hd; e += BLOCK) {
        float v = part[e];
        for (int g0 = 0; g0 < n_grp; g0 += 8) {                    // (ngrp: a multiple of 8; eight reads in flight, added in order)
            float t[8];
#pragma unroll
            for (int g = 0; g < 8; ++g) t[g] = part[(g0 + g) * hd + e];
#pragma unroll
            for (int g = 0; g < 8; ++g) if (g0 + g) v += t[g];
        }
        if (n_grp < ngrp) v += 0.0f;
        if (out_lds) { out_lds[e] = __float2half_rn(v); continue; }
        out[(size_t)h * hd + e] = v;
        if (out16) out16[out16_ol ? pi_ol_index(y, h * hd + e) : (size_t)h * hd + e] = __float2half_rn(v);
        if (q8_q) {                                               // (hd % 32 == 0: the lanes of a block run this together)
            float amax = fabsf(v);
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, PI_WAVE));
            const float d = pi_round_f16(pi_div(amax, 127.0f)), id = (amax != 0.0f) ? pi_div(127.0f, amax) : 0.0f;
            const int q = (int)rintf(__fmul_rn(v, id));
            int sq = q;
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) sq += __shfl_xor(sq, o, PI_WAVE);
            const int i = h * hd + e, eb = i & 31, t = y;
            q8_q[(((size_t)(i >> 5) * 4 + ((eb & 15) >> 2)) * 16 + t) * 8 + (eb >> 4) * 4 + (eb & 3)] = (int8_t)q;
            if (eb == 0) { q8_d[(size_t)(i >> 5) * 16 + t] = d; q8_s[(size_t)(i >> 5) * 16 + t] = -8 * sq; }
        }
    }
}

// ---------------------------------------------------------------------------------------------------
// Attention of one token with the cache cells of a head split over several workgroups (grid: head x part x sequence).  A compute unit
// pulls about 1/256 of the chip's HBM rate, so one workgroup per head leaves the K / V rows of a long context to 32 or 128 units
// (18 us per 7B layer at 600 cells, growing by 2.4 us per 100 cells); with n_parts workgroups per head every unit takes a share and
// the score buffer in LDS holds n_ctx / n_parts cells instead of all of them.
// Part s owns cells [n_kv * s / n, n_kv * (s + 1) / n); the last part holds the new cell: it rotates and stores k, stores v, and
// uses them from LDS.  Every part rotates q, computes its scores, e_i = fp16(exp(fp16(s_i - m))) with ITS maximum m (the rounding
// points of the CPU path's table, ggml.c:10747-10759), l = sum e_i in double and acc = sum v_i * e_i, and hands (m, l, acc) to
// attn_merge_kernel, which rescales by exp(m - M), adds the parts in order and divides by the total.  Against one workgroup per head,
// which knows the global maximum before it rounds, results differ in the last places of the fp16 roundings (1e-4 of the output).
// Bound by the trips to memory of a part's rows.  A group of lanes holds a cell's rows, the same cells of keys and values, so nothing but the maximum
// passes between groups before their sums meet.  Eight cells of a group, K and V, are on their way at any time, requested without a guard (a
// guarded load makes the compiler wait for all the others; past the last cell its rows are read again), and what the rotation
// needs ahead of them, because loads return in order.  Merge included, against the same sums with guarded loads and the soft-max of the whole workgroup
// between two barriers: 32 heads of 128 in 8 parts, 1030 cells 12.4 -> 11.0 us, 3001 19.4 -> 16.4 (49 MB), 32000 in 16 parts 97 -> 93.5; 128
// heads of 64 in 2 parts, 1030 cells 14.2 -> 12.3; 64 heads of 8 in 8 parts 17.5 -> 17.1, of 16 14.7 -> 14.2 (25.6 and 18.0 with what their 512 or 256 groups leave read one by one).
// ---------------------------------------------------------------------------------------------------
// FROM_CACHE: the token's own K / V row is in the cache already and qkv holds its rotated q only ([n_head * hd] per token; a prompt chunk
// behind rope_kv_store_kernel): nothing is rotated or stored, every cell is read from the cache.
constexpr int kAttnPartBlock = 512;
constexpr int kAttnPartCells = 4;        // cells of a group that are requested and used together; two such batches are in flight
// HERE: another workgroup of this launch reads the results.
template <bool FROM_CACHE, int LPP, bool HERE = false>
__device__ __forceinline__ void attn_part_head(const float * __restrict__ qkv, const float2 * __restrict__ rope_table,
                                                                   __half * __restrict__ k_cache, __half * __restrict__ v_cache,
                                                                   int n_head, int n_head_kv, int hd, int mode, int n_ctx, int s_cap,
                                                                   const int32_t * __restrict__ pos_p, float * __restrict__ part_acc, float * __restrict__ part_ml,
                                                                   int qkv_stride, size_t cache_seq_stride, const int h, const int sp, const int n_parts, const int z) {
    qkv += (size_t)z * qkv_stride;
    k_cache += (size_t)z * cache_seq_stride;
    v_cache += (size_t)z * cache_seq_stride;
    pos_p += z;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lpp = LPP ? LPP : hd / 8, ngrp = kAttnPartBlock / lpp;
    // sums of e_i and maxima, of the groups (32 or 64 of them: read at once) or, of the many groups of small heads and where their number is not a constant, of the waves
    constexpr int N = LPP ? kAttnPartBlock / LPP : kAttnPartBlock / PI_WAVE;
    __shared__ double sums[N];
    __shared__ float  tops[N];
    float * part = reinterpret_cast<float *>(smem);               // [ngrp][hd]
    float * qs   = part + kAttnPartBlock * 8;                     // [hd] rotated q, rounded to fp16
    float * kcur = qs + hd;                                       // [hd] rotated k of this position, rounded to fp16
    float * vcur = kcur + hd;                                     // [hd]
    float * s    = vcur + hd;                                     // [s_cap] scores of this part
    const int grp_sz = n_head / n_head_kv, kvh = h / grp_sz;
    const int tid = threadIdx.x;
    const int pos = *pos_p, n_kv = pos + 1;
    const int lo = (int)((long long)n_kv * sp / n_parts), hi = (int)((long long)n_kv * (sp + 1) / n_parts);
    const bool owns_new = !FROM_CACHE && sp == n_parts - 1;        // hi == n_kv: the new cell is this part's last
    const size_t slot = ((size_t)z * n_head + h) * n_parts + sp;
    if (hi - lo > s_cap) return;                                  // cannot happen for pos < n_ctx (the launcher sizes s_cap); never write past LDS
    const float * qsrc = qkv + (size_t)h * hd;
    const int sub = tid % lpp, grp = tid / lpp;
    const int n_old = (owns_new ? hi - 1 : hi) - lo;              // cells of this part that live in the cache
    // what is rotated: pair (or value) tid of the head, every thread one
    float q0 = 0, q1 = 0, k0 = 0, k1 = 0, v0 = 0;
    float2 cs{1, 0};
    const int pair = tid % (hd / 2), i0 = (mode & 2) ? pair : 2 * pair, i1 = (mode & 2) ? pair + hd / 2 : 2 * pair + 1;
    if constexpr (FROM_CACHE) q0 = qsrc[tid % hd];
    else {
        const float * ksrc = qkv + (size_t)(n_head + kvh) * hd, * vsrc = ksrc + (size_t)n_head_kv * hd;
        cs = rope_table[(size_t)pos * (hd / 2) + pair];
        q0 = qsrc[i0]; q1 = qsrc[i1]; k0 = ksrc[i0]; k1 = ksrc[i1]; v0 = vsrc[tid % hd];
    }
    const __half * kr = k_cache + ((size_t)kvh * n_ctx + lo) * hd + sub * 8, * vr = v_cache + ((size_t)kvh * n_ctx + lo) * hd + sub * 8;
    pi_u32x4 kk[2][kAttnPartCells], vv[2][kAttnPartCells];
    auto fetch = [&](pi_u32x4 * dst, const __half * rows, int c0) {
#pragma unroll
        for (int u = 0; u < kAttnPartCells; ++u) dst[u] = pi_ld16(rows + (size_t)max(min(c0 + u * ngrp + grp, n_old - 1), 0) * hd);
    };
    const int step = kAttnPartCells * ngrp;
    __builtin_amdgcn_sched_barrier(0);
    fetch(kk[0], kr, 0); fetch(kk[1], kr, step);
    fetch(vv[0], vr, 0); fetch(vv[1], vr, step);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FROM_CACHE) {
        if (tid < hd) qs[tid] = pi_round_f16(q0);
    } else {
        if (tid < hd / 2) {
            qs[i0] = pi_round_f16(__fsub_rn(__fmul_rn(q0, cs.x), __fmul_rn(q1, cs.y)));
            qs[i1] = pi_round_f16(__fadd_rn(__fmul_rn(q0, cs.y), __fmul_rn(q1, cs.x)));
        }
        if (owns_new && tid < hd) {
            const bool store = (h % grp_sz) == 0;
            const size_t cell = ((size_t)kvh * n_ctx + pos) * hd;
            if (tid < hd / 2) {
                const __half ka = __float2half_rn(__fsub_rn(__fmul_rn(k0, cs.x), __fmul_rn(k1, cs.y)));
                const __half kc = __float2half_rn(__fadd_rn(__fmul_rn(k0, cs.y), __fmul_rn(k1, cs.x)));
                kcur[i0] = __half2float(ka); kcur[i1] = __half2float(kc);
                if (store) { k_cache[cell + i0] = ka; k_cache[cell + i1] = kc; }
            }
            const __half v = __float2half_rn(v0);
            vcur[tid] = __half2float(v);
            if (store) v_cache[cell + tid] = v;
        }
    }
    __syncthreads();

    const float scale = pi_inv_sqrt((float)hd);
    float qf[8], top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) qf[i] = qs[sub * 8 + i];
    // the two batches in turn; f(which, first cell) uses a batch, then its registers are requested again for the next cells but one
    auto through = [&](pi_u32x4 (*regs)[kAttnPartCells], const __half * rows, auto && f) {
        for (int c0 = 0; c0 < n_old; c0 += 2 * step) {
            f(regs[0], c0);
            if (c0 + step >= n_old) break;
            fetch(regs[0], rows, c0 + 2 * step);
            f(regs[1], c0 + step);
            fetch(regs[1], rows, c0 + 3 * step);
        }
    };
    through(kk, kr, [&](const pi_u32x4 * k, int c0) {
#pragma unroll
        for (int u = 0; u < kAttnPartCells; ++u) {
            const int c = c0 + u * ngrp + grp;
            const float d = __fmul_rn(pi_group_sum<LPP>(pi_dot8(k[u], qf, 0.0f), lpp), scale);
            if (c < n_old) { top = fmaxf(top, d); if (sub == 0) s[c] = d; }
        }
    });
    const bool mine = owns_new && grp == n_old % ngrp;              // the new cell is this group's last
    if (mine) {
        float d = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) d = fmaf(kcur[sub * 8 + k], qf[k], d);
        d = __fmul_rn(pi_group_sum<LPP>(d, lpp), scale);
        top = fmaxf(top, d);
        if (sub == 0) s[n_old] = d;
    }
    const int slot_of = LPP ? grp : tid / PI_WAVE, lane_of = LPP ? sub : tid & (PI_WAVE - 1);
    if (!LPP) for (int o = lpp; o < PI_WAVE; o <<= 1) top = fmaxf(top, __shfl_xor(top, o, PI_WAVE));
    if (lane_of == 0) tops[slot_of] = top;
    __syncthreads();
    float mx = -INFINITY;
    for (int g = 0; g < N; g += 8)
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, tops[g + j]);

    float acc[8];
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    auto weight = [&](int c) { return pi_round_f16(expf(pi_round_f16(__fsub_rn(s[c], mx)))); };
    through(vv, vr, [&](const pi_u32x4 * v, int c0) {
        float e[kAttnPartCells];
#pragma unroll
        for (int u = 0; u < kAttnPartCells; ++u) e[u] = weight(min(c0 + u * ngrp + grp, n_old - 1));
#pragma unroll
        for (int u = 0; u < kAttnPartCells; ++u) {
            float vf[8];
            pi_unpack8(v[u], vf);
            if (c0 + u * ngrp + grp < n_old) {
                sum += (double)e[u];
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[k] = fmaf(vf[k], e[u], acc[k]);
            }
        }
    });
    if (mine) {
        const float e = weight(n_old);
        sum += (double)e;
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] = fmaf(vcur[sub * 8 + k], e, acc[k]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) part[grp * hd + sub * 8 + i] = acc[i];
    if (!LPP) for (int o = lpp; o < PI_WAVE; o <<= 1) sum += __shfl_xor(sum, o, PI_WAVE);       // (whole numbers of 2^-24: exact in any order)
    if (lane_of == 0) sums[slot_of] = sum;
    __syncthreads();
    const auto put = [](float * p, float v) {
        if constexpr (HERE) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *p = v;
    };
    if (tid < hd) {
        float v = part[tid];
        for (int g0 = 0; g0 < ngrp; g0 += 8) {                     // (ngrp: a multiple of 8; eight reads in flight, added in order)
            float t[8];
#pragma unroll
            for (int g = 0; g < 8; ++g) t[g] = part[(g0 + g) * hd + tid];
#pragma unroll
            for (int g = 0; g < 8; ++g) if (g0 + g) v += t[g];
        }
        put(part_acc + slot * hd + tid, v);
    } else if (tid == hd) {
        double l = 0.0;
        for (int g = 0; g < N; g += 8)
#pragma unroll
            for (int j = 0; j < 8; ++j) l += sums[g + j];
        put(part_ml + slot * 2, mx); put(part_ml + slot * 2 + 1, (float)l);
    }
}

// out[e] = sum_s acc_s[e] * exp(m_s - M) / sum_s l_s * exp(m_s - M) of a head, parts in ascending order.  HERE: the parts are results of other workgroups of this launch.
template <bool HERE>
__device__ __forceinline__ float attn_merge_value(const float * part_acc, const float * part_ml, int n_parts, int hd, size_t slot0, int e) {
    const auto get = [](const float * p) {
        if constexpr (HERE) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else return *p;
    };
    constexpr int kAtOnce = 16;                                    // parts whose values are requested together
    float m[kAtOnce], l[kAtOnce], a[kAtOnce], M = -INFINITY;
    auto fetch = [&](int s0, bool values) {
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
            const int sp = min(s0 + j, n_parts - 1);
            m[j] = get(part_ml + (slot0 + sp) * 2); l[j] = get(part_ml + (slot0 + sp) * 2 + 1);
            if (values) a[j] = get(part_acc + (slot0 + sp) * hd + e);
        }
    };
    fetch(0, true);
    for (int s0 = 0;;) {
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) M = fmaxf(M, m[j]);        // (the last part more than once)
        if ((s0 += kAtOnce) >= n_parts) break;
        fetch(s0, false);
    }
    if (n_parts > kAtOnce) fetch(0, true);
    float L = 0.0f, v = 0.0f;
    for (int s0 = 0;;) {
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j)
            if (s0 + j < n_parts && l[j] > 0.0f) {
                const float w = expf(__fsub_rn(m[j], M));
                L = fmaf(l[j], w, L);
                v = fmaf(a[j], w, v);
            }
        if ((s0 += kAtOnce) >= n_parts) break;
        fetch(s0, true);
    }
    return pi_div(v, L);
}

// LDS of attn_fused_kernel: the scores of every cell, one partial output row per group of hd/8 lanes, and q, k, v of the new cell
inline bool attn_fused_geometry_ok(int hd) {
    return hd > 0 && hd % 8 == 0 && (kAttnBlock / 2) % (hd / 8) == 0 && PI_WAVE % (hd / 8) == 0 && hd / 2 + hd <= kAttnBlock / 2;
}
inline size_t attn_fused_lds_bytes(int hd, int n_ctx, int block = kAttnBlock) {
    return sizeof(float) * ((size_t)n_ctx + (size_t)(block / (hd / 8)) * hd + 3 * (size_t)hd);
}
// and of attn_part_kernel
inline size_t attn_part_lds(int hd, int s_cap) { return sizeof(float) * ((size_t)s_cap + kAttnPartBlock * 8 + 3 * (size_t)hd); }

}  // namespace
