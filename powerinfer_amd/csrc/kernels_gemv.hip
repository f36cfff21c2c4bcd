// Mat-vecs of one token (fp16 and Q4_0 rows, fused norm prologue, ReLU / residual epilogues), embedding rows, greedy argmax, the
// random fills of synthetic models, and the workspace of the pi_k_* launchers.  gfx950, wave64.  Citations are file:line into the
// reference tree.
#include "kernels_common.hpp"

namespace {

// ---------------------------------------------------------------------------------------------------
// Dense F16 mat-vec.  A fixed grid of about two workgroups per CU (what a pure streaming read needs to reach
// HBM speed on this chip), each wave walking row groups g = wave_id, wave_id + n_waves, ...  A group is RPW
// consecutive rows; lane l reads 16 B (8 halfs) at column 8*l + 512*c of each row (chunk c), i.e. 1 KiB
// contiguous per row per load instruction.  The (group, chunk) space of a wave is flattened into steps of U
// chunks with one step of loads always in flight; the first step is issued before the activations are
// staged (weights do not depend on them).  Fast path: cols % 512 == 0 and rows % RPW == 0 (no guards).
// TAG only separates instantiations by role so that kernel traces can tell them apart.
// ---------------------------------------------------------------------------------------------------
constexpr int kGemvBlocks = 512;
constexpr int kFirstMostCols = 1024;   // widest vectors that stage_x_f16 holds in registers

template <int RPW, int U, int TAG>
__global__ __launch_bounds__(kBlock) void gemv_f16_kernel(const __half * __restrict__ W, const float * __restrict__ x, NormArgs na,
                                                          int epi, const float * add1, const float * add2,
                                                          float * __restrict__ y, int rows, int cols) {
    extern __shared__ __align__(16) unsigned char smem[];
    float * lds = reinterpret_cast<float *>(smem);
    __half * xs = reinterpret_cast<__half *>(smem + (size_t)cols * 8);
    __shared__ double red[16];

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n_waves = gridDim.x * kWavesPerBlock, wid = blockIdx.x * kWavesPerBlock + wave;
    const int n_groups = rows / RPW;
    const int spg = cols / (PI_WAVE * 8 * U);                              // steps per group
    const int my_groups = wid < n_groups ? (n_groups - wid + n_waves - 1) / n_waves : 0;
    const int T = my_groups * spg;

    stage_fast_issue(lds, x, na, cols);

    pi_u32x4 buf[RPW][U], nxt[RPW][U];
    const __half * wp = W + (size_t)wid * RPW * cols + lane * 8;           // this wave's position in the (group, step) walk
    int sig = 0;                                                           // step within the current group
    auto issue = [&](pi_u32x4 (&dst)[RPW][U]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < RPW; ++i) dst[i][u] = pi_ld_stream(wp + (size_t)i * cols + u * (PI_WAVE * 8));
        wp += U * PI_WAVE * 8;
        if (++sig == spg) { sig = 0; wp += (size_t)(n_waves * RPW - 1) * cols; }   // next group: (n_waves*RPW) rows down, back to column 0
    };
    if (T > 0) issue(buf);
    // the direct-to-LDS loads were issued first and complete in order: allow only the weight loads to remain in flight
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(RPW * U) : "memory");
    __syncthreads();
    stage_fast_finish(xs, lds, na, cols, red);

    float acc[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) acc[i] = 0.0f;
    int row = wid * RPW, c = lane * 8, s_in = 0;
    for (int t = 0; t < T; ++t) {
        if (t + 1 < T) issue(nxt);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float xf[8];
            pi_unpack8(pi_ld16(xs + c + u * (PI_WAVE * 8)), xf);
#pragma unroll
            for (int i = 0; i < RPW; ++i) acc[i] = pi_dot8(buf[i][u], xf, acc[i]);
        }
        c += U * PI_WAVE * 8;
        if (++s_in == spg) {
#pragma unroll
            for (int i = 0; i < RPW; ++i) {
                const float sum = pi_wave_sum(acc[i]);
                if (lane == 0) y[row + i] = apply_epilogue(sum, epi, add1, add2, row + i);
                acc[i] = 0.0f;
            }
            s_in = 0; c = lane * 8; row += n_waves * RPW;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < RPW; ++i) buf[i][u] = nxt[i][u];
    }
}

// state: the token loop's state, written where the host names the token (embed_start); token is then null
struct TokenStart { int32_t token, pos; int32_t * d_token, * d_pos, * d_step; };
__device__ __forceinline__ int32_t start_token(const int32_t * token, const TokenStart & s) {
    if (token) return __builtin_amdgcn_readfirstlane(*token);      // (in scalar registers, and no merge of the two reads through an address on the stack)
    if (blockIdx.x == 0 && threadIdx.x == 0) { *s.d_token = s.token; *s.d_pos = s.pos; *s.d_step = 0; }
    return s.token;
}
__global__ void resume_token_kernel(const float * __restrict__ row, int cols, TokenStart start, float * __restrict__ x) {
    start_token(nullptr, start);
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < cols) x[c] = row[c];
}
// The embedding row a mat-vec takes as its input: what a token begins with is no launch of its own where the first layer's q|k|v reads the row itself
// and its first workgroup leaves it in fp32 for the residual (and the state, see TokenStart).
struct EmbedRow { const void * table; const int32_t * token; TokenStart start; float * x; };
__device__ __forceinline__ float q4_value(const pi_block_q4_0 * b, int j) {
    uint16_t dbits; __builtin_memcpy(&dbits, &b->d, 2);
    const int q = (j < 16) ? (b->qs[j] & 0x0F) : (b->qs[j - 16] >> 4);
    return __fmul_rn((float)(q - 8), pi_f16_from_bits(dbits));
}
// eight columns from o on (a multiple of 8), stored by the first workgroup
template <bool Q4>
__device__ __forceinline__ void embed_eight(const EmbedRow & e, int32_t token, int cols, int o, float * v) {
    if (Q4) {
        const pi_block_q4_0 * b = (const pi_block_q4_0 *)e.table + (size_t)token * (cols / 32) + (o >> 5);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = q4_value(b, (o & 31) + k);
    } else {
        pi_unpack8(pi_ld16((const __half *)e.table + (size_t)token * cols + o), v);
    }
    if (blockIdx.x == 0) {
        *reinterpret_cast<float4 *>(e.x + o) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(e.x + o + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// Register-resident variant for cols == 512 * NCH (4096, 5120, 8192): a wave owns whole rows
// (row = wave_id, wave_id + n_waves, ...), lane l holds the activations of columns 8*l + 512*j as packed fp16 in
// registers, so the row loop touches neither LDS nor a workgroup barrier.  The prologue is shared by the four
// waves of a workgroup: wave w loads and normalises chunks w, w+4, ... of the vector (statistics cross the waves
// through LDS in wave order), the packed fp16 result meets in LDS and every wave reads all of it back once.
// 16 weight loads of 16 B per lane are in flight throughout (two rows, or the two halves of a wide row) and
// are issued before the prologue starts.  The residual operands of the epilogue travel with the row.
// KIND: 0 no norm, 1 RMSNorm * w, 2 LayerNorm * w + b.  TAG only names the role in kernel traces.
// MULTI: up to three matrices of the same width against the one vector in a single launch (the q, k and v projections of a host
// that keeps them as separate tensors): row r of the launch is row r of the first matrix, or row r - rows[0] of the second, ...
struct GemvMulti { const __half * W[3]; float * y[3]; int rows[3]; };
// STRIP: a workgroup owns kStripRows neighbouring rows and adds what a sparse FFN's workgroups left for them (out = FFN + W x + residual, the sums of ffn_reduce_kernel in its
// order).  Those vectors travel under the weights, and a launch behind this one is saved.  Workgroups with halves of a 128-byte line share a die.
constexpr int kStripRows = 16;
struct StripSum { const float * partial; int n_part; const uint32_t * words; int n_words; int32_t * n_active; const float * resid; };
template <int NCH, int KIND, bool MULTI, bool FIRST = false, bool STRIP = false>
__device__ __forceinline__ void gemv_f16_reg_body(const __half * __restrict__ W, const float * __restrict__ x,
                                                  const float * __restrict__ nw, const float * __restrict__ nb, float eps,
                                                  int epi, const float * __restrict__ add1, const float * __restrict__ add2,
                                                  float * __restrict__ y, int rows, const GemvMulti & mm, const EmbedRow & first = {}, const int blk = blockIdx.x, const int n_blk = gridDim.x, const StripSum & strip = {}) {
    constexpr int cols = NCH * 512;
    auto row_base = [&](int r) -> const __half * {
        if (!MULTI) return W + (size_t)r * cols;
        if (r < mm.rows[0]) return mm.W[0] + (size_t)r * cols;
        r -= mm.rows[0];
        if (r < mm.rows[1]) return mm.W[1] + (size_t)r * cols;
        return mm.W[2] + (size_t)(r - mm.rows[1]) * cols;
    };
    auto out_ptr = [&](int r) -> float * {
        if (!MULTI) return y + r;
        if (r < mm.rows[0]) return mm.y[0] + r;
        r -= mm.rows[0];
        if (r < mm.rows[1]) return mm.y[1] + r;
        return mm.y[2] + (r - mm.rows[1]);
    };
    constexpr bool kWide = NCH > 8;               // wide rows: the two buffers hold the halves of one row
    constexpr int CPB = kWide ? NCH / 2 : NCH;
    static_assert(!kWide || NCH % 2 == 0, "wide rows are split in two halves");
    constexpr int MYCH = (NCH + kWavesPerBlock - 1) / kWavesPerBlock;      // chunks a wave normalises
    __shared__ __align__(16) __half xs[cols];
    __shared__ double red[2][kWavesPerBlock];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int first_row = STRIP ? ((blk & 7) * (n_blk >> 3) + (blk >> 3)) * kStripRows : 0;
    const int n_waves = STRIP ? kWavesPerBlock : n_blk * kWavesPerBlock, wid = STRIP ? first_row + wave : blk * kWavesPerBlock + wave;
    const int end = STRIP ? first_row + kStripRows : rows;
    pi_u32x4 buf[2][CPB];
    float r1[2] = {0.0f, 0.0f}, r2[2] = {0.0f, 0.0f};
    auto issue = [&](int b, int r) {
        if (r < end) {
            const __half * wp = row_base(r) + lane * 8 + (kWide ? b * CPB * 512 : 0);
#pragma unroll
            for (int j = 0; j < CPB; ++j) buf[b][j] = pi_ld_stream(wp + j * 512);
            if (!kWide || b == 0) {
                if (epi >= PI_EPI_ADD) r1[b] = add1[r];
                if (epi == PI_EPI_ADD2) r2[b] = add2[r];
            }
        }
    };
    constexpr int kStripSlots = 64, kStripAhead = 4;              // vectors of workgroups slot, slot + 64, ...: four lanes have a strip's columns
    static_assert(!STRIP || kBlock == 4 * kStripSlots, "a slot is four lanes");
    const int slot = threadIdx.x >> 2;
    float4 ffn[STRIP ? kStripAhead : 1];
    float resid = 0.0f;
    int count = 0;
    __shared__ float dots[STRIP ? kStripRows : 1], tops[STRIP ? 8 : 1][kStripRows];
    issue(0, wid);
    issue(1, kWide ? wid : wid + n_waves);

    // ---- shared prologue ---------------------------------------------------------------------------------
    {
        float xv[MYCH][8], wv[MYCH][8], bv[MYCH][8];
        const int32_t token = FIRST ? start_token(first.token, first.start) : 0;
#pragma unroll
        for (int i = 0; i < MYCH; ++i) {
            const int j = wave + i * kWavesPerBlock;
            if (j < NCH) {
                const int o = j * 512 + lane * 8;
                if (FIRST) embed_eight<false>(first, token, cols, o, xv[i]);
                else {
                    const float4 a = *reinterpret_cast<const float4 *>(x + o), b = *reinterpret_cast<const float4 *>(x + o + 4);
                    xv[i][0] = a.x; xv[i][1] = a.y; xv[i][2] = a.z; xv[i][3] = a.w; xv[i][4] = b.x; xv[i][5] = b.y; xv[i][6] = b.z; xv[i][7] = b.w;
                }
                if (KIND >= 1) {
                    const float4 c = *reinterpret_cast<const float4 *>(nw + o), e = *reinterpret_cast<const float4 *>(nw + o + 4);
                    wv[i][0] = c.x; wv[i][1] = c.y; wv[i][2] = c.z; wv[i][3] = c.w; wv[i][4] = e.x; wv[i][5] = e.y; wv[i][6] = e.z; wv[i][7] = e.w;
                }
                if (KIND == 2) {
                    const float4 c = *reinterpret_cast<const float4 *>(nb + o), e = *reinterpret_cast<const float4 *>(nb + o + 4);
                    bv[i][0] = c.x; bv[i][1] = c.y; bv[i][2] = c.z; bv[i][3] = c.w; bv[i][4] = e.x; bv[i][5] = e.y; bv[i][6] = e.z; bv[i][7] = e.w;
                }
            }
        }
        if constexpr (STRIP) {
#pragma unroll
            for (int u = 0; u < kStripAhead; ++u) {
                const int p = slot + u * kStripSlots;
                ffn[u] = *reinterpret_cast<const float4 *>(strip.partial + (size_t)(p < strip.n_part ? p : slot) * cols + first_row + (threadIdx.x & 3) * 4);
            }
            if (threadIdx.x < kStripRows) resid = strip.resid[first_row + threadIdx.x];
            if (blk == 0) for (int w = threadIdx.x; w < strip.n_words; w += kBlock) count += __popc(strip.words[w]);
        }
        float mean = 0.0f, scale = 1.0f;
        if (KIND >= 1) {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < MYCH; ++i)
                if (wave + i * kWavesPerBlock < NCH) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) s += KIND == 1 ? (double)__fmul_rn(xv[i][k], xv[i][k]) : (double)xv[i][k];
                }
            s = pi_wave_sum_f64(s);
            if (lane == 0) red[0][wave] = s;
            __syncthreads();
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < kWavesPerBlock; ++w) t += red[0][w];
            if (KIND == 1) scale = pi_inv_sqrt((float)(t / cols) + eps);
            else {
                mean = (float)(t / cols);
                double s2 = 0.0;
#pragma unroll
                for (int i = 0; i < MYCH; ++i)
                    if (wave + i * kWavesPerBlock < NCH) {
#pragma unroll
                        for (int k = 0; k < 8; ++k) { const float v = __fsub_rn(xv[i][k], mean); s2 += (double)__fmul_rn(v, v); }
                    }
                s2 = pi_wave_sum_f64(s2);
                if (lane == 0) red[1][wave] = s2;
                __syncthreads();
                double t2 = 0.0;
#pragma unroll
                for (int w = 0; w < kWavesPerBlock; ++w) t2 += red[1][w];
                scale = pi_inv_sqrt((float)(t2 / cols) + eps);
            }
        }
#pragma unroll
        for (int i = 0; i < MYCH; ++i) {
            const int j = wave + i * kWavesPerBlock;
            if (j < NCH) {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    float v = xv[i][k];
                    if (KIND >= 1) v = __fmul_rn(__fmul_rn(KIND == 2 ? __fsub_rn(v, mean) : v, scale), wv[i][k]);
                    if (KIND == 2) v = __fadd_rn(v, bv[i][k]);
                    xv[i][k] = v;
                }
                __half2 hh[4] = {__floats2half2_rn(xv[i][0], xv[i][1]), __floats2half2_rn(xv[i][2], xv[i][3]),
                                 __floats2half2_rn(xv[i][4], xv[i][5]), __floats2half2_rn(xv[i][6], xv[i][7])};
                *reinterpret_cast<pi_u32x4 *>(xs + j * 512 + lane * 8) = *reinterpret_cast<const pi_u32x4 *>(hh);
            }
        }
        __syncthreads();
    }
    pi_u32x4 xr[NCH];
#pragma unroll
    for (int j = 0; j < NCH; ++j) xr[j] = *reinterpret_cast<const pi_u32x4 *>(xs + j * 512 + lane * 8);

    auto finish = [&](float acc, float a1, float a2, int r) {
        acc = pi_wave_sum(acc);
        if (epi == PI_EPI_RELU) acc = fmaxf(acc, 0.0f);
        else if (epi == PI_EPI_ADD) acc = __fadd_rn(acc, a1);
        else if (epi == PI_EPI_ADD2) acc = __fadd_rn(__fadd_rn(acc, a1), a2);
        if constexpr (STRIP) { if (lane == 0) dots[r - first_row] = acc; }
        else if (lane == 0) *out_ptr(r) = acc;
    };
    if constexpr (kWide) {
        for (int r = wid; r < end; r += n_waves) {
            // keep the activations packed: widening them once outside the loop would double their register footprint
#pragma unroll
            for (int j = 0; j < NCH; ++j) asm volatile("" : "+v"(xr[j].x), "+v"(xr[j].y), "+v"(xr[j].z), "+v"(xr[j].w));
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < CPB; ++j) acc = pi_dot8h(buf[0][j], xr[j], acc);
            const float a1 = r1[0], a2 = r2[0];
            issue(0, r + n_waves);
#pragma unroll
            for (int j = 0; j < CPB; ++j) acc = pi_dot8h(buf[1][j], xr[CPB + j], acc);
            issue(1, r + n_waves);
            finish(acc, a1, a2, r);
        }
    } else {
        for (int r = wid; r < end; r += 2 * n_waves) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int rr = r + b * n_waves;
                if (rr < end) {
                    float acc = 0.0f;
#pragma unroll
                    for (int j = 0; j < NCH; ++j) acc = pi_dot8h(buf[b][j], xr[j], acc);
                    finish(acc, r1[b], r2[b], rr);
                }
                issue(b, rr + 2 * n_waves);
            }
        }
    }
    if constexpr (STRIP) {
        float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const auto add = [&](const float4 & v) { sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w; };
#pragma unroll
        for (int u = 0; u < kStripAhead; ++u) if (slot + u * kStripSlots < strip.n_part) add(ffn[u]);
        for (int p = slot + kStripAhead * kStripSlots; p < strip.n_part; p += kStripSlots) add(*reinterpret_cast<const float4 *>(strip.partial + (size_t)p * cols + first_row + (threadIdx.x & 3) * 4));
#pragma unroll
        for (int o = 4; o < 32; o <<= 1) {                          // eight slots
            sum.x += __shfl_xor(sum.x, o, PI_WAVE); sum.y += __shfl_xor(sum.y, o, PI_WAVE); sum.z += __shfl_xor(sum.z, o, PI_WAVE); sum.w += __shfl_xor(sum.w, o, PI_WAVE);
        }
        if ((lane & 31) < 4) *reinterpret_cast<float4 *>(&tops[wave * 2 + (lane >> 5)][(lane & 3) * 4]) = sum;
        if (blk == 0) { count = pi_wave_sum_i32(count); if (lane == 0) red[0][wave] = count; }
        __syncthreads();
        if (threadIdx.x < kStripRows) {
            float f = tops[0][threadIdx.x];
#pragma unroll
            for (int g = 1; g < 8; ++g) f += tops[g][threadIdx.x];
            y[first_row + threadIdx.x] = __fadd_rn(__fadd_rn(f, dots[threadIdx.x]), resid);
        }
        if (blk == 0 && threadIdx.x == 0 && strip.n_active) *strip.n_active = (int)(red[0][0] + red[0][1] + red[0][2] + red[0][3]);
    }
}

template <int NCH, int KIND, int TAG>
__global__ __launch_bounds__(kBlock, 2) void gemv_f16_reg_kernel(const __half * __restrict__ W, const float * __restrict__ x,
                                                              const float * __restrict__ nw, const float * __restrict__ nb, float eps,
                                                              int epi, const float * __restrict__ add1, const float * __restrict__ add2,
                                                              float * __restrict__ y, int rows) {
    gemv_f16_reg_body<NCH, KIND, false>(W, x, nw, nb, eps, epi, add1, add2, y, rows, GemvMulti{});
}
template <int NCH, int KIND>
__global__ __launch_bounds__(kBlock, 2) void gemv_f16_first_kernel(const __half * __restrict__ W, EmbedRow first, const float * __restrict__ nw, const float * __restrict__ nb, float eps,
                                                                  float * __restrict__ y, int rows) {
    gemv_f16_reg_body<NCH, KIND, false, true>(W, nullptr, nw, nb, eps, PI_EPI_NONE, nullptr, nullptr, y, rows, GemvMulti{}, first);
}
// A mat-vec and the sums of a sparse FFN's vectors.  Bound by HBM: 134 MB of weights and 8 MB of vectors in 25.0 us (5.7 TB/s); as two launches 22.9 + 4.8 and the gap between
// them.  Falcon-40B shapes, 8 tokens of 4 layers: 4680 -> 4620 us at 1024 cells, 4780 -> 4690 at 100.
template <int NCH>
__global__ __launch_bounds__(kBlock, 2) void gemv_strip_f16_kernel(const __half * __restrict__ W, const float * __restrict__ x, float * __restrict__ y, StripSum strip) {
    gemv_f16_reg_body<NCH, 0, false, false, true>(W, x, nullptr, nullptr, 0.0f, PI_EPI_NONE, nullptr, nullptr, y, NCH * 512, GemvMulti{}, EmbedRow{}, blockIdx.x, gridDim.x, strip);
}
// Two matrices of one vector, the second one without a norm and with a ReLU: workgroups in proportion to their rows.  Bound by HBM: 9216 + 1024 rows of 8192 columns, 168 MB
// in 28.5 us (5.9 TB/s).
template <int NCH, int KIND>
__global__ __launch_bounds__(kBlock, 2) void gemv_pair_f16_reg_kernel(const __half * __restrict__ W, const float * __restrict__ x, const float * __restrict__ nw, const float * __restrict__ nb, float eps,
                                                                     float * __restrict__ y, int rows, int blocks, const __half * __restrict__ W2, float * __restrict__ y2, int rows2) {
    if ((int)blockIdx.x < blocks) gemv_f16_reg_body<NCH, KIND, false>(W, x, nw, nb, eps, PI_EPI_NONE, nullptr, nullptr, y, rows, GemvMulti{}, EmbedRow{}, blockIdx.x, blocks);
    else gemv_f16_reg_body<NCH, 0, false>(W2, x, nullptr, nullptr, 0.0f, PI_EPI_RELU, nullptr, nullptr, y2, rows2, GemvMulti{}, EmbedRow{}, (int)blockIdx.x - blocks, (int)gridDim.x - blocks);
}
template <int NCH, int KIND>
__global__ __launch_bounds__(kBlock, 2) void gemv_multi_f16_reg_kernel(GemvMulti mm, const float * __restrict__ x,
                                                                    const float * __restrict__ nw, const float * __restrict__ nb, float eps, int rows) {
    gemv_f16_reg_body<NCH, KIND, true>(nullptr, x, nw, nb, eps, PI_EPI_NONE, nullptr, nullptr, nullptr, rows, mm);
}

// ---------------------------------------------------------------------------------------------------
// Q4_0 mat-vec for cols == 4096 * CB.  A Q4_0 row of 4096 weights is 128 blocks of 18 bytes = 2304 bytes = 64 lanes x 36 bytes: lane l
// meets the block pair (2l, 2l+1) of each 4096-column group with the matching 64 int8 activations, their two Q8_0 scales and block sums,
// all held in registers.  The nibbles are used unsigned through v_dot4_i32_i8 and 8 * sum(x) is subtracted per block, which is exact in
// int32; the result is scaled by d_w * d_x in fp32 as vec_dot_q4_0_q8_0 does (ggml-quants.c:2512-2650).  The prologue (norm, then Q8_0
// quantisation as the x86 quantize_row_q8_0 does: d = amax / 127 kept as fp16, q = rint(x * 127 / amax), ggml-quants.c:702-760) is
// shared by the four waves through LDS.
// A fifth wave copies rows straight to LDS, a row for each of the other four a step and NBUF steps ahead, from the first moment on: the matrix
// is on its way under the prologue, which is half of the launch, and a lane takes its 36 bytes from LDS, where 36 bytes a lane fall on
// different banks (from memory they were three loads at odd places each).  One barrier a step: behind it the step's rows are there and
// the previous step's slots are free.  12288 x 4096 behind an RMSNorm 10.8 -> 9.7 us, 32000 x 4096 20.2 -> 16.1,
// 8192 x 8192 12.6 -> 9.1, 65024 x 8192 69 -> 54 (5.5 TB/s).
// OFF: a matrix on a multiple of 4 bytes only.  Its rows are copied from the multiple of 16 before them, one piece more, and the lanes read that
// much further on (the 16 bytes around its first and last byte lie on their page): 10.8 -> 9.9, 20.1 -> 16.1, 12.7 -> 9.4, 70 -> 57 us
// (copied by single words: 32000 x 4096 21.6).
// ---------------------------------------------------------------------------------------------------
constexpr int kQ4Threads = kBlock + PI_WAVE;
template <int CB, int KIND, bool OFF, bool FIRST>
__device__ __forceinline__ void gemv_q4_reg_body(const unsigned char * __restrict__ W, const float * __restrict__ x,
                                                 const float * __restrict__ nw, const float * __restrict__ nb, float eps,
                                                 int epi, const float * __restrict__ add1, const float * __restrict__ add2,
                                                 float * __restrict__ y, int rows, const EmbedRow & first) {
    constexpr int cols = CB * 4096, NCH = cols / 512, nblk = cols / 32;
    constexpr int NBUF = CB == 1 ? 5 : 2;                          // steps in LDS
    constexpr int MYCH = NCH / kWavesPerBlock;
    constexpr size_t row_bytes = (size_t)nblk * 18;
    __shared__ __align__(16) int8_t xq[cols];
    __shared__ float xd[nblk];
    __shared__ int   xsum[nblk];
    __shared__ double red[2][kWavesPerBlock];
    __shared__ __align__(16) unsigned char ring[NBUF][kWavesPerBlock][row_bytes + (OFF ? 16 : 0)];
    const int mis = OFF ? (int)((uintptr_t)W & 15) : 0;            // a multiple of 4; rows are multiples of 16
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n_waves = gridDim.x * kWavesPerBlock, wid = blockIdx.x * kWavesPerBlock + wave;

    const int steps = (rows - 1 - (int)blockIdx.x * kWavesPerBlock) / n_waves + 1;         // (of the first wave: the others' may be one fewer)
    if (wave == kWavesPerBlock) {
        constexpr int kCopies = kWavesPerBlock * (int)((row_bytes + 1023) / 1024);         // of a step
        static_assert((NBUF - 1) * kCopies <= 63, "the counter of loads in flight");
        typedef const __attribute__((address_space(1))) void * gptr;
        typedef __attribute__((address_space(3))) void * lptr;
        auto copy_step = [&](int s) {
#pragma unroll
            for (int w = 0; w < kWavesPerBlock; ++w) {
                const unsigned char * p = W + (size_t)min((int)blockIdx.x * kWavesPerBlock + w + s * n_waves, rows - 1) * row_bytes;
                unsigned char * to = ring[s % NBUF][w];
#pragma unroll
                for (int o = 0; o < (int)row_bytes; o += 1024)
                    if (o + 1024 <= (int)row_bytes || o + lane * 16 < (int)row_bytes + mis) __builtin_amdgcn_global_load_lds((gptr)(p - mis + o + lane * 16), (lptr)(to + o), 16, 0, 0);
            }
        };
        for (int s = 0; s < min(steps, NBUF); ++s) copy_step(s);
        for (int k = 0; k <= KIND; ++k) __builtin_amdgcn_s_barrier();                      // the prologue's
        for (int s = 0; s < steps; ++s) {
            const int behind = min(steps - 1 - s, s ? NBUF - 2 : NBUF - 1);               // steps on their way behind this one (step s - 1's slot is filled below)
            if (behind == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else if (behind == 1) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kCopies) : "memory");
            else if (behind == 2) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NBUF > 2 ? 2 * kCopies : 0) : "memory");
            else if (behind == 3) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NBUF > 3 ? 3 * kCopies : 0) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NBUF > 4 ? 4 * kCopies : 0) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (s > 0 && s - 1 + NBUF < steps) copy_step(s - 1 + NBUF);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // no copy may arrive in LDS that is no longer this workgroup's
        return;
    }

    // ---- shared prologue: norm, Q8_0 quantisation -------------------------------------------------------------
    {
        float xv[MYCH][8], wv[MYCH][8], bv[MYCH][8];
        const int32_t token = FIRST ? start_token(first.token, first.start) : 0;
#pragma unroll
        for (int i = 0; i < MYCH; ++i) {
            const int o = (wave + i * kWavesPerBlock) * 512 + lane * 8;
            if (FIRST) embed_eight<true>(first, token, cols, o, xv[i]);
            else {
                const float4 a = *reinterpret_cast<const float4 *>(x + o), b = *reinterpret_cast<const float4 *>(x + o + 4);
                xv[i][0] = a.x; xv[i][1] = a.y; xv[i][2] = a.z; xv[i][3] = a.w; xv[i][4] = b.x; xv[i][5] = b.y; xv[i][6] = b.z; xv[i][7] = b.w;
            }
            if (KIND >= 1) {
                const float4 c = *reinterpret_cast<const float4 *>(nw + o), e = *reinterpret_cast<const float4 *>(nw + o + 4);
                wv[i][0] = c.x; wv[i][1] = c.y; wv[i][2] = c.z; wv[i][3] = c.w; wv[i][4] = e.x; wv[i][5] = e.y; wv[i][6] = e.z; wv[i][7] = e.w;
            }
            if (KIND == 2) {
                const float4 c = *reinterpret_cast<const float4 *>(nb + o), e = *reinterpret_cast<const float4 *>(nb + o + 4);
                bv[i][0] = c.x; bv[i][1] = c.y; bv[i][2] = c.z; bv[i][3] = c.w; bv[i][4] = e.x; bv[i][5] = e.y; bv[i][6] = e.z; bv[i][7] = e.w;
            }
        }
        float mean = 0.0f, scale = 1.0f;
        if (KIND >= 1) {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < MYCH; ++i)
#pragma unroll
                for (int k = 0; k < 8; ++k) s += KIND == 1 ? (double)__fmul_rn(xv[i][k], xv[i][k]) : (double)xv[i][k];
            s = pi_wave_sum_f64(s);
            if (lane == 0) red[0][wave] = s;
            __syncthreads();
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < kWavesPerBlock; ++w) t += red[0][w];
            if (KIND == 1) scale = pi_inv_sqrt((float)(t / cols) + eps);
            else {
                mean = (float)(t / cols);
                double s2 = 0.0;
#pragma unroll
                for (int i = 0; i < MYCH; ++i)
#pragma unroll
                    for (int k = 0; k < 8; ++k) { const float v = __fsub_rn(xv[i][k], mean); s2 += (double)__fmul_rn(v, v); }
                s2 = pi_wave_sum_f64(s2);
                if (lane == 0) red[1][wave] = s2;
                __syncthreads();
                double t2 = 0.0;
#pragma unroll
                for (int w = 0; w < kWavesPerBlock; ++w) t2 += red[1][w];
                scale = pi_inv_sqrt((float)(t2 / cols) + eps);
            }
        }
#pragma unroll
        for (int i = 0; i < MYCH; ++i) {
            const int j = wave + i * kWavesPerBlock;
            float amax = 0.0f;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float v = xv[i][k];
                if (KIND >= 1) v = __fmul_rn(__fmul_rn(KIND == 2 ? __fsub_rn(v, mean) : v, scale), wv[i][k]);
                if (KIND == 2) v = __fadd_rn(v, bv[i][k]);
                xv[i][k] = v;
                amax = fmaxf(amax, fabsf(v));
            }
            // a quad of lanes holds one block of 32 values
            amax = fmaxf(amax, pi_dpp_f32<PI_DPP_XOR1, 0xF>(amax));
            amax = fmaxf(amax, pi_dpp_f32<PI_DPP_XOR2, 0xF>(amax));
            const float d = pi_div(amax, 127.0f);
            const float id = (amax != 0.0f) ? pi_div(127.0f, amax) : 0.0f;
            int q[8], qs = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) { q[k] = (int)rintf(__fmul_rn(xv[i][k], id)); qs += q[k]; }
            qs += pi_dpp_i32<PI_DPP_XOR1, 0xF>(qs);
            qs += pi_dpp_i32<PI_DPP_XOR2, 0xF>(qs);
            const uint32_t p0 = (uint32_t)(q[0] & 0xff) | ((uint32_t)(q[1] & 0xff) << 8) | ((uint32_t)(q[2] & 0xff) << 16) | ((uint32_t)(q[3] & 0xff) << 24);
            const uint32_t p1 = (uint32_t)(q[4] & 0xff) | ((uint32_t)(q[5] & 0xff) << 8) | ((uint32_t)(q[6] & 0xff) << 16) | ((uint32_t)(q[7] & 0xff) << 24);
            *reinterpret_cast<pi_u32x2 *>(xq + j * 512 + lane * 8) = pi_u32x2{p0, p1};
            if ((lane & 3) == 0) { xd[j * 16 + (lane >> 2)] = pi_round_f16(d); xsum[j * 16 + (lane >> 2)] = qs; }
        }
        __syncthreads();
    }
    int   X[CB][16];
    float dx[CB][2];
    int   sx[CB][2];
#pragma unroll
    for (int g = 0; g < CB; ++g) {
        const int b0 = g * 128 + 2 * lane;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const pi_u32x4 v = *reinterpret_cast<const pi_u32x4 *>(xq + b0 * 32 + k * 16);
            X[g][4 * k] = (int)v.x; X[g][4 * k + 1] = (int)v.y; X[g][4 * k + 2] = (int)v.z; X[g][4 * k + 3] = (int)v.w;
        }
        dx[g][0] = xd[b0]; dx[g][1] = xd[b0 + 1];
        sx[g][0] = xsum[b0]; sx[g][1] = xsum[b0 + 1];
    }

    for (int s = 0; s < steps; ++s) {
        const int rr = wid + s * n_waves;
        float r1 = 0.0f, r2 = 0.0f;
        if (rr < rows) {
            if (epi >= PI_EPI_ADD) r1 = add1[rr];
            if (epi == PI_EPI_ADD2) r2 = add2[rr];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // the last step's row has been read
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (rr >= rows) continue;
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < CB; ++g) {
            uint32_t d9[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) d9[k] = *reinterpret_cast<const uint32_t *>(ring[s % NBUF][wave] + mis + g * 2304 + lane * 36 + k * 4);
            int s0 = 0, s1 = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t q0 = __builtin_amdgcn_alignbit(d9[k + 1], d9[k], 16);       // bytes 2 + 4k .. 5 + 4k of the pair
                s0 = __builtin_amdgcn_sdot4((int)(q0 & 0x0F0F0F0Fu), X[g][k], s0, false);
                s0 = __builtin_amdgcn_sdot4((int)((q0 >> 4) & 0x0F0F0F0Fu), X[g][4 + k], s0, false);
                const uint32_t q1 = d9[5 + k];
                s1 = __builtin_amdgcn_sdot4((int)(q1 & 0x0F0F0F0Fu), X[g][8 + k], s1, false);
                s1 = __builtin_amdgcn_sdot4((int)((q1 >> 4) & 0x0F0F0F0Fu), X[g][12 + k], s1, false);
            }
            s0 -= 8 * sx[g][0];
            s1 -= 8 * sx[g][1];
            acc = fmaf(__fmul_rn(pi_f16_from_bits((uint16_t)(d9[0] & 0xffffu)), dx[g][0]), (float)s0, acc);
            acc = fmaf(__fmul_rn(pi_f16_from_bits((uint16_t)(d9[4] >> 16)), dx[g][1]), (float)s1, acc);
        }
        acc = pi_wave_sum(acc);
        if (epi == PI_EPI_RELU) acc = fmaxf(acc, 0.0f);
        else if (epi == PI_EPI_ADD) acc = __fadd_rn(acc, r1);
        else if (epi == PI_EPI_ADD2) acc = __fadd_rn(__fadd_rn(acc, r1), r2);
        if (lane == 0) y[rr] = acc;
    }
}

template <int CB, int KIND, int TAG, bool OFF>
__global__ __launch_bounds__(kQ4Threads, 2) void gemv_q4_reg_kernel(const unsigned char * __restrict__ W, const float * __restrict__ x,
                                                             const float * __restrict__ nw, const float * __restrict__ nb, float eps,
                                                             int epi, const float * __restrict__ add1, const float * __restrict__ add2,
                                                             float * __restrict__ y, int rows) {
    gemv_q4_reg_body<CB, KIND, OFF, false>(W, x, nw, nb, eps, epi, add1, add2, y, rows, EmbedRow{});
}
template <int CB, int KIND, bool OFF>
__global__ __launch_bounds__(kQ4Threads, 2) void gemv_q4_first_kernel(const unsigned char * __restrict__ W, EmbedRow first, const float * __restrict__ nw, const float * __restrict__ nb,
                                                                     float eps, float * __restrict__ y, int rows) {
    gemv_q4_reg_body<CB, KIND, OFF, true>(W, nullptr, nw, nb, eps, PI_EPI_NONE, nullptr, nullptr, y, rows, first);
}

// Any shape with cols % 8 == 0: one wave per row, grid-stride.  Short rows are bound by latency: the input's round trip and its norm, then
// the row's.  The first row's first 2048 columns are therefore requested before the input is staged (clamped addresses: a load under a branch
// of its own would be waited for before the next): with the input held in registers, 3.75 -> 3.35 us at 512 columns and 512..1536 rows.
struct HalfRow { const __half * p; __device__ __forceinline__ float operator[](int i) const { return __half2float(p[i]); } };
template <bool FIRST>
__device__ __forceinline__ void gemv_f16_generic_body(const __half * __restrict__ W, const float * __restrict__ x, NormArgs na,
                                                      int epi, const float * add1, const float * add2,
                                                      float * __restrict__ y, int rows, int cols, const EmbedRow & embed) {
    extern __shared__ __align__(16) unsigned char smem[];
    __half * xs = reinterpret_cast<__half *>(smem);
    __shared__ double red[16];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int r = blockIdx.x * kWavesPerBlock + wave;
    constexpr int kFirst = 4;
    pi_u32x4 first[kFirst];
    const __half * w0 = W + (size_t)min(r, rows - 1) * cols;
#pragma unroll
    for (int u = 0; u < kFirst; ++u) first[u] = pi_ld_stream(w0 + min((u * PI_WAVE + lane) * 8, cols - 8));
    if (FIRST) {
        const HalfRow row{(const __half *)embed.table + (size_t)start_token(embed.token, embed.start) * cols};
        if (blockIdx.x == 0) for (int i = threadIdx.x; i < cols; i += kBlock) embed.x[i] = row[i];
        stage_x_f16(xs, row, cols, na, red);
    } else {
        stage_x_f16(xs, x, cols, na, red);
    }
    bool held = true;
    for (; r < rows; r += gridDim.x * kWavesPerBlock) {
        float acc = 0.0f;
        int c = lane * 8;
        if (held) {
            held = false;
#pragma unroll
            for (int u = 0; u < kFirst; ++u, c += PI_WAVE * 8)
                if (c < cols) {
                    float xf[8];
                    pi_unpack8(pi_ld16(xs + c), xf);
                    acc = pi_dot8(first[u], xf, acc);
                }
        }
#pragma unroll 4
        for (; c < cols; c += PI_WAVE * 8) {
            float xf[8];
            pi_unpack8(pi_ld16(xs + c), xf);
            acc = pi_dot8(pi_ld_stream(W + (size_t)r * cols + c), xf, acc);
        }
        acc = pi_wave_sum(acc);
        if (lane == 0) y[r] = apply_epilogue(acc, epi, add1, add2, r);
    }
}
__global__ __launch_bounds__(kBlock) void gemv_f16_generic_kernel(const __half * __restrict__ W, const float * __restrict__ x, NormArgs na,
                                                                  int epi, const float * add1, const float * add2,
                                                                  float * __restrict__ y, int rows, int cols) {
    gemv_f16_generic_body<false>(W, x, na, epi, add1, add2, y, rows, cols, EmbedRow{});
}
__global__ __launch_bounds__(kBlock) void gemv_f16_generic_first_kernel(const __half * __restrict__ W, EmbedRow first, NormArgs na, float * __restrict__ y, int rows, int cols) {
    gemv_f16_generic_body<true>(W, nullptr, na, PI_EPI_NONE, nullptr, nullptr, y, rows, cols, first);
}


// Dense Q4_0 mat-vec: one wave per RPW rows, lane l owns blocks l, l+64, ...
template <int RPW>
__global__ __launch_bounds__(kBlock) void gemv_q4_kernel(const pi_block_q4_0 * __restrict__ W, const float * __restrict__ x, NormArgs na,
                                                         int epi, const float * add1, const float * add2,
                                                         float * __restrict__ y, int rows, int cols) {
    extern __shared__ __align__(16) unsigned char smem[];
    int8_t * xq   = reinterpret_cast<int8_t *>(smem);
    float  * xd   = reinterpret_cast<float *>(smem + cols);
    float  * xtmp = reinterpret_cast<float *>(smem + cols + (cols / 32) * 4);
    __shared__ double red[16];
    stage_x_q8(xq, xd, x, cols, na, red, xtmp);

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nb = cols / 32;
    const int n_groups = (rows + RPW - 1) / RPW;
    for (int g = blockIdx.x * kWavesPerBlock + wave; g < n_groups; g += gridDim.x * kWavesPerBlock) {
        const int r0 = g * RPW;
        float acc[RPW];
#pragma unroll
        for (int i = 0; i < RPW; ++i) acc[i] = 0.0f;
        for (int b = lane; b < nb; b += PI_WAVE) {
            const float dx = xd[b];
#pragma unroll
            for (int i = 0; i < RPW; ++i)
                if (r0 + i < rows) acc[i] = q4_block_dot(W + (size_t)(r0 + i) * nb + b, xq + b * 32, dx, acc[i]);
        }
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            const float s = pi_wave_sum(acc[i]);
            if (lane == 0 && r0 + i < rows) y[r0 + i] = apply_epilogue(s, epi, add1, add2, r0 + i);
        }
    }
}

__global__ void embed_f16_kernel(const __half * __restrict__ table, int cols, const int32_t * __restrict__ token, float * __restrict__ x, TokenStart start) {
    const __half * row = table + (size_t)start_token(token, start) * cols;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < cols; i += gridDim.x * blockDim.x) x[i] = __half2float(row[i]);
}
// blockIdx.y = token of a chunk (0 for a single token)
__global__ void embed_q4_kernel(const pi_block_q4_0 * __restrict__ table, int cols, const int32_t * __restrict__ token, float * __restrict__ x, TokenStart start) {
    const pi_block_q4_0 * row = table + (size_t)start_token(token ? token + blockIdx.y : nullptr, start) * (cols / 32);
    x += (size_t)blockIdx.y * cols;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < cols; i += gridDim.x * blockDim.x) {
        x[i] = q4_value(row + (i >> 5), i & 31);
    }
}
// Rows of a chunk's tokens, which travel as the kernel's arguments: copying 130 of them and their positions to the device and waiting for the copies took
// 31 us ahead of a prompt's first product (a prompt of 131: 1913 -> 1882 us).  Eight values a thread; wide: rows and x on 16 bytes.
struct ChunkTokens { static constexpr int kMost = 512; int32_t id[kMost]; };
template <bool Q4>
__global__ __launch_bounds__(256) void embed_chunk_kernel(const void * __restrict__ table, int cols, ChunkTokens tokens, int pos0, float * __restrict__ x, int32_t * __restrict__ pos, int wide) {
    const int t = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (blockIdx.x == 0 && threadIdx.x == 0) pos[t] = pos0 + t;
    if (c >= cols) return;
    float v[8];
    if (Q4) {
        const pi_block_q4_0 * b = (const pi_block_q4_0 *)table + (size_t)tokens.id[t] * (cols / 32) + c / 32;
        uint16_t dbits; __builtin_memcpy(&dbits, &b->d, 2);
        const float d = pi_f16_from_bits(dbits);
        const int j = c & 15, high = c & 16 ? 4 : 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = __fmul_rn((float)(((b->qs[j + k] >> high) & 0x0F) - 8), d);
    } else {
        const __half * row = (const __half *)table + (size_t)tokens.id[t] * cols + c;
        if (wide) {
            const pi_u32x4 raw = *reinterpret_cast<const pi_u32x4 *>(row);
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = pi_f16_from_bits((uint16_t)(w[k / 2] >> (16 * (k & 1))));
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = c + k < cols ? __half2float(row[k]) : 0.0f;
        }
    }
    float * o = x + (size_t)t * cols + c;
    if (wide) {
        *reinterpret_cast<float4 *>(o) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(o + 4) = make_float4(v[4], v[5], v[6], v[7]);
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) if (c + k < cols) o[k] = v[k];
    }
}

// first maximum wins (std::max_element, llama.cpp:8617-8631)
__global__ __launch_bounds__(1024) void argmax_kernel(const float * __restrict__ logits, int n, int32_t * __restrict__ token_out) {
    __shared__ float bv[16];
    __shared__ int   bi[16];
    float best = -INFINITY; int idx = 0x7fffffff;
    for (int i = threadIdx.x; i < n; i += blockDim.x) { const float v = logits[i]; if (v > best) { best = v; idx = i; } }
    if (idx == 0x7fffffff) { idx = n; }                          // thread saw nothing above -inf
#pragma unroll
    for (int o = PI_WAVE / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, PI_WAVE); const int oi = __shfl_xor(idx, o, PI_WAVE);
        if (ov > best || (ov == best && oi < idx)) { best = ov; idx = oi; }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { bv[wave] = best; bi[wave] = idx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
            if (bv[w] > best || (bv[w] == best && bi[w] < idx)) { best = bv[w]; idx = bi[w]; }
        *token_out = idx < n ? idx : 0;
    }
}

// counter-based N(0, std^2): two 32-bit hashes -> Box-Muller; deterministic in (seed, index)
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__global__ void fill_normal_f16_kernel(__half * __restrict__ p, size_t n, uint64_t seed, float std, const float * __restrict__ row_bias, int cols) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint64_t r = mix64(seed * 0xD1342543DE82EF95ull + i);
        const float u1 = ((uint32_t)(r >> 32) + 1.0f) * (1.0f / 4294967296.0f);
        const float u2 = (uint32_t)r * (1.0f / 4294967296.0f);
        float v = sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2) * std;
        if (row_bias) v += row_bias[i / cols];
        p[i] = __float2half_rn(v);
    }
}

// the same values rounded to bf16
__global__ void fill_normal_bf16_kernel(__bf16 * __restrict__ p, size_t n, uint64_t seed, float std) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint64_t r = mix64(seed * 0xD1342543DE82EF95ull + i);
        const float u1 = ((uint32_t)(r >> 32) + 1.0f) * (1.0f / 4294967296.0f);
        const float u2 = (uint32_t)r * (1.0f / 4294967296.0f);
        p[i] = (__bf16)(sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2) * std);
    }
}

// N(0, std^2) values quantised to Q4_0 exactly as quantize_row_q4_0_reference does (ggml-quants.c:428-463): the
// element of largest magnitude (first one wins) sets d = max / -8, q = min(15, (int)(x / d + 8.5)).  One thread per block.
__global__ void fill_normal_q4_0_kernel(pi_block_q4_0 * __restrict__ p, size_t n_blocks, uint64_t seed, float std) {
    for (size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x; b < n_blocks; b += (size_t)gridDim.x * blockDim.x) {
        float v[32];
        float amax = 0.0f, mx = 0.0f;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint64_t r = mix64(seed * 0xD1342543DE82EF95ull + b * 32 + j);
            const float u1 = ((uint32_t)(r >> 32) + 1.0f) * (1.0f / 4294967296.0f);
            const float u2 = (uint32_t)r * (1.0f / 4294967296.0f);
            v[j] = pi_round_f16(sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2) * std);
            if (fabsf(v[j]) > amax) { amax = fabsf(v[j]); mx = v[j]; }
        }
        const float d = mx / -8.0f;
        const float id = d != 0.0f ? pi_div(1.0f, d) : 0.0f;
        pi_block_q4_0 blk;
        blk.d = pi_f16_bits(d);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int q0 = min(15, (int)(v[j] * id + 8.5f)), q1 = min(15, (int)(v[j + 16] * id + 8.5f));
            blk.qs[j] = (uint8_t)(q0 | (q1 << 4));
        }
        p[b] = blk;
    }
}

}  // namespace

extern "C" {

pi_workspace * pi_workspace_create(int max_ff, int max_d) {
    if (max_ff <= 0 || max_d <= 0 || (max_d + kAxpyTile - 1) / kAxpyTile > 62) { pi::set_error("pi_workspace_create: bad sizes"); return nullptr; }
    pi_workspace * ws = new pi_workspace{};
    ws->max_ff = max_ff; ws->max_d = max_d;
    const size_t n_words = (size_t)(max_ff / 32 + 2) > 2048 ? (size_t)(max_ff / 32 + 2) : 2048;       // groups of 32 neurons, or two words per compute unit
    ws->words    = (uint32_t *)pi_malloc(sizeof(uint32_t) * n_words);
    ws->words_hot = (uint32_t *)pi_malloc(sizeof(uint32_t) * (max_ff / 32 + 2));
    ws->counters = (unsigned int *)pi_malloc(sizeof(unsigned int) * 64);
    ws->partial  = (float *)pi_malloc(sizeof(float) * (size_t)kAxpyGroups * max_d);
    ws->hq       = (int32_t *)pi_malloc(sizeof(int32_t) * max_ff);
    ws->hd       = (float *)pi_malloc(sizeof(float) * max_ff);
    const size_t n_part = (size_t)((max_ff + 31) / 32) > (size_t)kBmGroups * kBtMaxT ? (size_t)((max_ff + 31) / 32) : (size_t)kBmGroups * kBtMaxT;
    ws->ffn_partial = (float *)pi_malloc(sizeof(float) * n_part * max_d);
    ws->hc_batch = (__half *)pi_malloc(sizeof(__half) * ((size_t)max_ff + 16) * kBtMaxT);
    ws->row_any = (unsigned char *)pi_malloc((size_t)max_ff + 16);
    if (!ws->words || !ws->words_hot || !ws->counters || !ws->partial || !ws->hq || !ws->hd || !ws->ffn_partial || !ws->hc_batch || !ws->row_any) {
        pi_workspace_destroy(ws); return nullptr;
    }
    pi_memset(ws->counters, 0, sizeof(unsigned int) * 64);
    return ws;
}
int pi_workspace_destroy(pi_workspace * ws) {
    if (!ws) return PI_OK;
    pi_free(ws->words); pi_free(ws->words_hot); pi_free(ws->counters); pi_free(ws->partial); pi_free(ws->hq); pi_free(ws->hd); pi_free(ws->ffn_partial); pi_free(ws->hc_batch); pi_free(ws->row_any);
    delete ws;
    return PI_OK;
}

int pi_k_gemv(int wtype, const void * W, int rows, int cols, const float * x, const pi_norm * norm,
              int epilogue, const float * add1, const float * add2, float * y, pi_stream_t stream) {
    if (!W || !x || !y || rows <= 0 || cols <= 0) return pi::fail(PI_E_ARG, "pi_k_gemv: null pointer or empty shape");
    if (epilogue < 0 || epilogue > PI_EPI_ADD2 || (epilogue >= PI_EPI_ADD && !add1) || (epilogue == PI_EPI_ADD2 && !add2))
        return pi::fail(PI_E_ARG, "pi_k_gemv: bad epilogue arguments");
    hipStream_t st = (hipStream_t)stream;
    const NormArgs na = to_norm(norm);
    // rows per wave group / chunks per step: 8 x 16 B loads in flight per lane per step, and at least one
    // group for each of the grid's waves
    const int n_waves = kGemvBlocks * kWavesPerBlock;
    const int rpw = rows >= 4 * n_waves ? 4 : rows >= 2 * n_waves ? 2 : 1;
    const int n_groups = (rows + rpw - 1) / rpw;
    int blocks = (n_groups + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks > kGemvBlocks) blocks = kGemvBlocks;
    if (wtype == PI_TYPE_F16) {
        if (cols % 8) return pi::fail(PI_E_ARG, "pi_k_gemv: F16 needs cols % 8 == 0");
        const __half * w = (const __half *)W;
        const int u = 8 / rpw;
        const bool fast = cols % (PI_WAVE * 8 * u) == 0 && rows % rpw == 0 && stage_fast_lds_bytes(cols) <= 64 * 1024 &&
                          (((uintptr_t)x | (uintptr_t)(norm ? norm->w : nullptr)) & 15) == 0;
        const bool aligned = (((uintptr_t)x | (uintptr_t)(norm ? norm->w : nullptr) | (uintptr_t)(norm ? norm->b : nullptr)) & 15) == 0;
        const int rblocks = rows >= n_waves ? kGemvBlocks : (rows + kWavesPerBlock - 1) / kWavesPerBlock;
        // register-resident kernel: the norm must carry what its kind needs (RMSNorm a weight, LayerNorm weight and bias)
        const bool reg_ok = aligned && (cols == 4096 || cols == 5120 || cols == 8192) &&
                            (na.kind == 0 || (na.kind == 1 && na.w && !na.b) || (na.kind == 2 && na.w && na.b));
        if (reg_ok) {
            // the tag only names the role in kernel traces: 1 = lm-head sized, 2 = fewer rows than the grid has waves
            const int tag = rows >= 16384 ? 1 : rows < n_waves ? 2 : 0;
#define PI_GEMV_REG(NCH, KIND, TAG) hipLaunchKernelGGL((gemv_f16_reg_kernel<NCH, KIND, TAG>), dim3(rblocks), dim3(kBlock), 0, st, w, x, na.w, na.b, na.eps, epilogue, add1, add2, y, rows)
#define PI_GEMV_REG_K(NCH, KIND) do { if (tag == 1) PI_GEMV_REG(NCH, KIND, 1); else if (tag == 2) PI_GEMV_REG(NCH, KIND, 2); else PI_GEMV_REG(NCH, KIND, 0); } while (0)
#define PI_GEMV_REG_N(NCH) do { if (na.kind == 0) PI_GEMV_REG_K(NCH, 0); else if (na.kind == 1) PI_GEMV_REG_K(NCH, 1); else PI_GEMV_REG_K(NCH, 2); } while (0)
            if (cols == 4096) PI_GEMV_REG_N(8); else if (cols == 5120) PI_GEMV_REG_N(10); else PI_GEMV_REG_N(16);
#undef PI_GEMV_REG_N
#undef PI_GEMV_REG_K
#undef PI_GEMV_REG
        } else if (fast) {
            const size_t sh = stage_fast_lds_bytes(cols);
            if (rows >= 16384) hipLaunchKernelGGL((gemv_f16_kernel<4, 2, 1>), dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
            else if (rpw == 4) hipLaunchKernelGGL((gemv_f16_kernel<4, 2, 0>), dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
            else if (rpw == 2) hipLaunchKernelGGL((gemv_f16_kernel<2, 4, 0>), dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
            else               hipLaunchKernelGGL((gemv_f16_kernel<1, 8, 0>), dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
        } else {
            const size_t sh = (size_t)cols * 2;
            if (sh > 60 * 1024) return pi::fail(PI_E_UNSUPPORTED, "pi_k_gemv: cols too large for LDS staging");
            int gb = (rows + kWavesPerBlock - 1) / kWavesPerBlock;
            if (gb > 2048) gb = 2048;
            hipLaunchKernelGGL(gemv_f16_generic_kernel, dim3(gb), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
        }
    } else if (wtype == PI_TYPE_Q4_0) {
        if (cols % 32) return pi::fail(PI_E_ARG, "pi_k_gemv: Q4_0 needs cols % 32 == 0");
        const size_t sh = (size_t)cols + (size_t)(cols / 32) * 4 + (size_t)cols * 4;
        if (sh > 60 * 1024) return pi::fail(PI_E_UNSUPPORTED, "pi_k_gemv: cols too large for LDS staging");
        const pi_block_q4_0 * w = (const pi_block_q4_0 *)W;
        const bool aligned = (((uintptr_t)x | (uintptr_t)(norm ? norm->w : nullptr) | (uintptr_t)(norm ? norm->b : nullptr)) & 15) == 0 && ((uintptr_t)W & 3) == 0;
        const bool reg_ok = aligned && (cols == 4096 || cols == 8192) &&
                            (na.kind == 0 || (na.kind == 1 && na.w && !na.b) || (na.kind == 2 && na.w && na.b));
        if (reg_ok) {
            const int rblocks = rows >= n_waves ? kGemvBlocks : (rows + kWavesPerBlock - 1) / kWavesPerBlock;
            const int tag = rows >= 16384 ? 1 : 0;
            const unsigned char * wb = (const unsigned char *)W;
#define PI_GEMV_Q4_O(CB, KIND, TAG, OFF) hipLaunchKernelGGL((gemv_q4_reg_kernel<CB, KIND, TAG, OFF>), dim3(rblocks), dim3(kQ4Threads), 0, st, wb, x, na.w, na.b, na.eps, epilogue, add1, add2, y, rows)
#define PI_GEMV_Q4(CB, KIND, TAG) do { if ((uintptr_t)W & 15) PI_GEMV_Q4_O(CB, KIND, TAG, true); else PI_GEMV_Q4_O(CB, KIND, TAG, false); } while (0)
#define PI_GEMV_Q4_K(CB, KIND) do { if (tag == 1) PI_GEMV_Q4(CB, KIND, 1); else PI_GEMV_Q4(CB, KIND, 0); } while (0)
#define PI_GEMV_Q4_N(CB) do { if (na.kind == 0) PI_GEMV_Q4_K(CB, 0); else if (na.kind == 1) PI_GEMV_Q4_K(CB, 1); else PI_GEMV_Q4_K(CB, 2); } while (0)
            if (cols == 4096) PI_GEMV_Q4_N(1); else PI_GEMV_Q4_N(2);
#undef PI_GEMV_Q4_N
#undef PI_GEMV_Q4_K
#undef PI_GEMV_Q4
#undef PI_GEMV_Q4_O
            return pi::check_launch("pi_k_gemv");
        }
        if (rpw == 8)      hipLaunchKernelGGL(gemv_q4_kernel<8>, dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
        else if (rpw == 4) hipLaunchKernelGGL(gemv_q4_kernel<4>, dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
        else if (rpw == 2) hipLaunchKernelGGL(gemv_q4_kernel<2>, dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
        else               hipLaunchKernelGGL(gemv_q4_kernel<1>, dim3(blocks), dim3(kBlock), sh, st, w, x, na, epilogue, add1, add2, y, rows, cols);
    } else {
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_gemv: weight type must be F16 or Q4_0");
    }
    return pi::check_launch("pi_k_gemv");
}

int pi_k_gemv_multi_f16(const void * const * W, const int * rows, int n_mat, int cols, const float * x, const pi_norm * norm, float * const * y,
                        pi_stream_t stream) {
    if (!W || !rows || !y || !x || n_mat < 1 || n_mat > 3) return pi::fail(PI_E_ARG, "pi_k_gemv_multi_f16: one to three matrices");
    const NormArgs na = to_norm(norm);
    GemvMulti mm{};
    int total = 0;
    for (int i = 0; i < 3; ++i) {
        if (i < n_mat) {
            if (!W[i] || !y[i] || rows[i] <= 0) return pi::fail(PI_E_ARG, "pi_k_gemv_multi_f16: null matrix or result, or no rows");
            mm.W[i] = (const __half *)W[i]; mm.y[i] = y[i]; mm.rows[i] = rows[i]; total += rows[i];
        }
    }
    const bool aligned = (((uintptr_t)x | (uintptr_t)na.w | (uintptr_t)na.b) & 15) == 0;
    if (!aligned || (cols != 4096 && cols != 5120 && cols != 8192) || !(na.kind == 0 || (na.kind == 1 && na.w && !na.b) || (na.kind == 2 && na.w && na.b)))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_gemv_multi_f16: cols 4096, 5120 or 8192, 16-byte aligned vectors, a norm that carries its weights");
    hipStream_t st = (hipStream_t)stream;
    const int n_waves = kGemvBlocks * kWavesPerBlock;
    const int rblocks = total >= n_waves ? kGemvBlocks : (total + kWavesPerBlock - 1) / kWavesPerBlock;
#define PI_GEMV_M(NCH, KIND) hipLaunchKernelGGL((gemv_multi_f16_reg_kernel<NCH, KIND>), dim3(rblocks), dim3(kBlock), 0, st, mm, x, na.w, na.b, na.eps, total)
#define PI_GEMV_M_N(NCH) do { if (na.kind == 0) PI_GEMV_M(NCH, 0); else if (na.kind == 1) PI_GEMV_M(NCH, 1); else PI_GEMV_M(NCH, 2); } while (0)
    if (cols == 4096) PI_GEMV_M_N(8); else if (cols == 5120) PI_GEMV_M_N(10); else PI_GEMV_M_N(16);
#undef PI_GEMV_M_N
#undef PI_GEMV_M
    return pi::check_launch("pi_k_gemv_multi_f16");
}

int pi_k_embed_batch_q4(const void * table_q4, int cols, const int32_t * tokens, int T, float * x, pi_stream_t stream) {
    if (!table_q4 || !tokens || !x || cols <= 0 || cols % 32 || T <= 0 || T > kChunkMaxT) return pi::fail(PI_E_ARG, "pi_k_embed_batch_q4: bad arguments");
    hipLaunchKernelGGL(embed_q4_kernel, dim3((cols + 255) / 256, T), dim3(256), 0, (hipStream_t)stream, (const pi_block_q4_0 *)table_q4, cols, tokens, x, TokenStart{});
    return pi::check_launch("pi_k_embed_batch_q4");
}

static int embed_one(int wtype, const void * table, int cols, const int32_t * token, const TokenStart & start, float * x, hipStream_t st) {
    const int blocks = (cols + 255) / 256;
    if (wtype == PI_TYPE_F16)       hipLaunchKernelGGL(embed_f16_kernel, dim3(blocks), dim3(256), 0, st, (const __half *)table, cols, token, x, start);
    else if (wtype == PI_TYPE_Q4_0) hipLaunchKernelGGL(embed_q4_kernel, dim3(blocks), dim3(256), 0, st, (const pi_block_q4_0 *)table, cols, token, x, start);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_embed: table type must be F16 or Q4_0");
    return pi::check_launch("pi_k_embed");
}

int pi_k_embed(int wtype, const void * table, int cols, const int32_t * token, float * x, pi_stream_t stream) {
    if (!table || !token || !x || cols <= 0) return pi::fail(PI_E_ARG, "pi_k_embed: bad arguments");
    return embed_one(wtype, table, cols, token, TokenStart{}, x, (hipStream_t)stream);
}

// W . norm(row of the embedding), for the widths of the mat-vecs that hold their input in registers and for what the kernel for any F16 shape takes.  Not for
// the others, whose input travels to LDS as it lies in memory.  A token's embedding launch was 2.1 to 2.9 us, and a gap, for a row that every
// workgroup of the next launch could read as well.  Eight tokens of a call each, us: 7B F16 3995 -> 3961, 7B Q4_0
// behind 2.8 k cells 3890 -> 3845; sixteen of three layers of 512 columns 1660 -> 1645.
int pi_k_first_gemv_supported(int wtype, const void * table, const void * W, int rows, int cols, const pi_norm * norm, const float * x) {
    const NormArgs na = to_norm(norm);
    if (!table || !W || !x || rows <= 0 || cols <= 0 || (((uintptr_t)x | (uintptr_t)na.w | (uintptr_t)na.b) & 15) || na.kind < 1 || na.kind > 2 || !na.w || (na.kind == 2) != (na.b != nullptr)) return 0;
    if (wtype == PI_TYPE_Q4_0) return (cols == 4096 || cols == 8192) && !((uintptr_t)W & 3);
    if (wtype != PI_TYPE_F16 || ((uintptr_t)table & 15) || cols % 8) return 0;
    return cols == 4096 || cols == 5120 || cols == 8192 || cols <= kFirstMostCols;
}
int pi_k_first_gemv(int wtype, const void * table, const int32_t * token, int32_t id, int32_t pos, int32_t * d_token, int32_t * d_pos, int32_t * d_step, const void * W, int rows, int cols,
               const pi_norm * norm, float * x, float * y, pi_stream_t stream) {
    if (!pi_k_first_gemv_supported(wtype, table, W, rows, cols, norm, x) || !y || (!token && (!d_token || !d_pos || !d_step))) return pi::fail(PI_E_ARG, "pi_k_first_gemv: bad arguments");
    hipStream_t st = (hipStream_t)stream;
    const NormArgs na = to_norm(norm);
    const EmbedRow first{table, token, {id, pos, d_token, d_pos, d_step}, x};
    const int full = (rows + kWavesPerBlock - 1) / kWavesPerBlock, blocks = std::min(full, kGemvBlocks);
    const bool layer = na.kind == 2, off = ((uintptr_t)W & 15) != 0;
#define PI_FIRST_F16(NCH, KIND) hipLaunchKernelGGL((gemv_f16_first_kernel<NCH, KIND>), dim3(blocks), dim3(kBlock), 0, st, (const __half *)W, first, na.w, na.b, na.eps, y, rows)
#define PI_FIRST_Q4(CB, KIND, OFF) hipLaunchKernelGGL((gemv_q4_first_kernel<CB, KIND, OFF>), dim3(blocks), dim3(kQ4Threads), 0, st, (const unsigned char *)W, first, na.w, na.b, na.eps, y, rows)
#define PI_FIRST_Q4_K(CB, KIND) do { if (off) PI_FIRST_Q4(CB, KIND, true); else PI_FIRST_Q4(CB, KIND, false); } while (0)
    if (wtype == PI_TYPE_Q4_0) {
        if (cols == 4096) { if (layer) PI_FIRST_Q4_K(1, 2); else PI_FIRST_Q4_K(1, 1); }
        else { if (layer) PI_FIRST_Q4_K(2, 2); else PI_FIRST_Q4_K(2, 1); }
    } else if (cols == 4096) { if (layer) PI_FIRST_F16(8, 2); else PI_FIRST_F16(8, 1); }
    else if (cols == 5120) { if (layer) PI_FIRST_F16(10, 2); else PI_FIRST_F16(10, 1); }
    else if (cols == 8192) { if (layer) PI_FIRST_F16(16, 2); else PI_FIRST_F16(16, 1); }
    else hipLaunchKernelGGL(gemv_f16_generic_first_kernel, dim3(std::min(full, 2048)), dim3(kBlock), (size_t)cols * 2, st, (const __half *)W, first, na, y, rows, cols);
#undef PI_FIRST_Q4_K
#undef PI_FIRST_Q4
#undef PI_FIRST_F16
    return pi::check_launch("pi_k_first_gemv");
}

}  // extern "C"
namespace pi {
int embed_start(int wtype, const void * table, int cols, int32_t token, int32_t pos, int32_t * d_token, int32_t * d_pos, int32_t * d_step, float * x, pi_stream_t stream) {
    if (!table || !d_token || !d_pos || !d_step || !x || cols <= 0) return fail(PI_E_ARG, "embed_start: bad arguments");
    return embed_one(wtype, table, cols, nullptr, TokenStart{token, pos, d_token, d_pos, d_step}, x, (hipStream_t)stream);
}
bool gemv_pair_supported(int type, int type2, int cols, const pi_norm * norm, const float * x) {
    const NormArgs na = to_norm(norm);
    return type == PI_TYPE_F16 && type2 == PI_TYPE_F16 && cols == 8192 && na.kind == 2 && na.w && na.b && (((uintptr_t)x | (uintptr_t)na.w | (uintptr_t)na.b) & 15) == 0;
}
int gemv_pair(const void * W, int rows, const pi_norm * norm, float * y, const void * W2, int rows2, float * y2, int cols, const float * x, pi_stream_t stream) {
    if (!W || !W2 || !x || !y || !y2 || rows <= 0 || rows2 <= 0 || !gemv_pair_supported(PI_TYPE_F16, PI_TYPE_F16, cols, norm, x)) return fail(PI_E_ARG, "gemv_pair: bad arguments");
    const NormArgs na = to_norm(norm);
    const long long all = (long long)rows + rows2;
    const int second = std::min(std::max((int)((kGemvBlocks * (long long)rows2 + all / 2) / all), 1), kGemvBlocks - 1);
    hipLaunchKernelGGL((gemv_pair_f16_reg_kernel<16, 2>), dim3(kGemvBlocks), dim3(kBlock), 0, (hipStream_t)stream, (const __half *)W, x, na.w, na.b, na.eps, y, rows, kGemvBlocks - second,
                       (const __half *)W2, y2, rows2);
    return check_launch("gemv_pair");
}
int gemv_ffn_out(const void * W, int cols, const float * x, const float * resid, float * y, int32_t * n_active, pi_workspace * ws, pi_stream_t stream) {
    if (!W || !x || !resid || !y || !ws || cols != 8192 || cols > ws->max_d || ((uintptr_t)x & 15)) return fail(PI_E_ARG, "gemv_ffn_out: bad arguments");
    if (ws->pf_parts < 64 || ws->pf_words <= 0 || ws->pf_words > ws->max_ff / 32 + 2048) return fail(PI_E_STATE, "gemv_ffn_out: no fused launch has filled this workspace");
    hipLaunchKernelGGL((gemv_strip_f16_kernel<16>), dim3(cols / kStripRows), dim3(kBlock), 0, (hipStream_t)stream, (const __half *)W, x, y,
                       StripSum{ws->ffn_partial, ws->pf_parts, ws->words, ws->pf_words, n_active, resid});
    return check_launch("gemv_ffn_out");
}
int resume_token(const float * row, int cols, int32_t token, int32_t pos, int32_t * d_token, int32_t * d_pos, int32_t * d_step, float * x, pi_stream_t stream) {
    if (!row || !d_token || !d_pos || !d_step || !x || cols <= 0) return fail(PI_E_ARG, "resume_token: bad arguments");
    hipLaunchKernelGGL(resume_token_kernel, dim3((cols + 255) / 256), dim3(256), 0, (hipStream_t)stream, row, cols, TokenStart{token, pos, d_token, d_pos, d_step}, x);
    return check_launch("resume_token");
}
int embed_chunk(int wtype, const void * table, int cols, const int32_t * tokens, int T, int pos, float * x, int32_t * d_pos, pi_stream_t stream) {
    const bool q4 = wtype == PI_TYPE_Q4_0;
    if (!table || !tokens || !x || !d_pos || cols <= 0 || T <= 0 || (q4 && cols % 32)) return fail(PI_E_ARG, "embed_chunk: bad arguments");
    if (!q4 && wtype != PI_TYPE_F16) return fail(PI_E_UNSUPPORTED, "embed_chunk: table type must be F16 or Q4_0");
    const int wide = cols % 8 == 0 && (((uintptr_t)x | (q4 ? 0 : (uintptr_t)table)) & 15) == 0;
    for (int t0 = 0; t0 < T; t0 += ChunkTokens::kMost) {
        const int n = T - t0 < ChunkTokens::kMost ? T - t0 : ChunkTokens::kMost;
        ChunkTokens ids{};
        for (int t = 0; t < n; ++t) ids.id[t] = tokens[t0 + t];
        hipLaunchKernelGGL(q4 ? embed_chunk_kernel<true> : embed_chunk_kernel<false>, dim3((cols + 2047) / 2048, n), dim3(256), 0, (hipStream_t)stream, table, cols, ids, pos + t0,
                           x + (size_t)t0 * cols, d_pos + t0, wide);
    }
    return check_launch("embed_chunk");
}
}  // namespace pi
extern "C" {

int pi_k_argmax(const float * logits, int n, int32_t * token_out, pi_stream_t stream) {
    if (!logits || !token_out || n <= 0) return pi::fail(PI_E_ARG, "pi_k_argmax: bad arguments");
    hipLaunchKernelGGL(argmax_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, logits, n, token_out);
    return pi::check_launch("pi_k_argmax");
}

int pi_fill_normal_f16(void * dptr, size_t n, uint64_t seed, float std, const float * row_bias, int cols, pi_stream_t stream) {
    if (!dptr || (row_bias && cols <= 0)) return pi::fail(PI_E_ARG, "pi_fill_normal_f16: bad arguments");
    if (n == 0) return PI_OK;
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_normal_f16_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (__half *)dptr, n, seed, std, row_bias, cols);
    return pi::check_launch("pi_fill_normal_f16");
}

int pi_fill_normal_bf16(void * dptr, size_t n, uint64_t seed, float std, pi_stream_t stream) {
    if (!dptr) return pi::fail(PI_E_ARG, "pi_fill_normal_bf16: null pointer");
    if (n == 0) return PI_OK;
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_normal_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (__bf16 *)dptr, n, seed, std);
    return pi::check_launch("pi_fill_normal_bf16");
}

int pi_fill_normal_q4_0(void * dptr, size_t n_weights, uint64_t seed, float std, pi_stream_t stream) {
    if (!dptr || n_weights % 32) return pi::fail(PI_E_ARG, "pi_fill_normal_q4_0: null pointer or a weight count that is not a multiple of 32");
    if (n_weights == 0) return PI_OK;
    size_t blocks = (n_weights / 32 + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_normal_q4_0_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (pi_block_q4_0 *)dptr, n_weights / 32, seed, std);
    return pi::check_launch("pi_fill_normal_q4_0");
}

}  // extern "C"
