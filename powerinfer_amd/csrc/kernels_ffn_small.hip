// The sparse FFN of one token in a small F16 model, predictor included: both of its products, the active rows and the down projection in one launch
// and a reduction, where wider models need the predictor's hidden units and the rows of one launch spread over the chip.
#include "kernels_common.hpp"
#include "runtime.hpp"
#include "../../include/powerinfer_hip.h"

namespace {

// A workgroup owns 32 neurons.  Every workgroup forms all R hidden units itself, then the logits of its neurons, which the waves hold eight each,
// and its share of gate, up and down rows: the active neurons are dealt to the four waves in turn, and a wave that has one holds whole rows of it,
// so nothing but the waves' partial outputs meets at the end.  Bound by what one unit can read: every 64 KB of fc1 are 2.2 us, about a launch by
// itself (with all of it in flight at once, with workgroups that begin at different rows and with the products on the matrix cores the times are the
// same within 5 %).  512 columns, 4096 neurons, rank 128, a tenth active: 7.6 us and 2.8 for the reduction, against 16.6 for four launches
// (predictor 2.9 + 3.5, gate and up 5.5, down 4.7); 16 tokens of such a model of three layers 2076 -> 1722 us.
// Rounding as in those: hidden units, normed input and h to fp16, everything else fp32; logits have the same order of sums.
// KIND: norm of the FFN's input (0 none, 1 RMS, 2 LayerNorm); the predictor reads x as it is.
constexpr int kSmBlock = 256, kSmNeurons = 32, kSmFc1 = 16, kSmAtOnce = 4;      // rows of fc1 in flight a wave; neurons whose rows a wave requests together
// SUM: x is what the heads' shares of the output projection make of it (attn_out_small_kernel), and the first workgroup leaves it for the residual.
template <int CH, int R, bool GATE, int KIND, bool SUM = false>      // columns: 512 CH
__global__ __launch_bounds__(kSmBlock) void ffn_small_f16_kernel(const __half * __restrict__ fc1, const __half * __restrict__ fc2, const __half * __restrict__ up, const __half * __restrict__ gate,
                                                                 const __half * __restrict__ down, const float * __restrict__ x, const float * __restrict__ nw, const float * __restrict__ nb,
                                                                 float eps, float thr, uint32_t * __restrict__ words, float * __restrict__ partial,
                                                                 const float * __restrict__ shares, int n_shares, float * __restrict__ xsum) {
    constexpr int COLS = 512 * CH, LPN = R / 8, NPL = 64 / LPN, NL = 8 / NPL, OWN = R / 4, HELD = kSmFc1 / CH, NB = OWN / HELD;
    static_assert(LPN == 8 || LPN == 16 || LPN == 32, "rank");
    __shared__ __align__(16) __half hid[R];
    __shared__ __align__(16) float part[4][COLS];
    __shared__ uint32_t word[4];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n0 = (int)blockIdx.x * kSmNeurons;
    float xv[CH][8], wv[CH][8], bv[CH][8];
    auto fetch8 = [&](float (&v)[8], const float * p) {
        const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    };
#pragma unroll
    for (int j = 0; j < CH; ++j) fetch8(xv[j], x + j * 512 + lane * 8);
    constexpr int kSmShares = 8;                                    // vectors a wave requests together
    float sv[SUM ? kSmShares : 1][CH][8];
    auto fetch_shares = [&](int s0) {                               // (past the last one its values again, not added)
#pragma unroll
        for (int s = 0; s < kSmShares; ++s)
#pragma unroll
            for (int j = 0; j < CH; ++j) fetch8(sv[s][j], shares + (size_t)min(s0 + s, n_shares - 1) * COLS + j * 512 + lane * 8);
    };
    if constexpr (SUM) fetch_shares(0);
    pi_u32x4 f1[2][HELD][CH], f2[NL];
    auto fetch1 = [&](pi_u32x4 (&f)[HELD][CH], int b) {
#pragma unroll
        for (int k = 0; k < HELD; ++k)
#pragma unroll
            for (int j = 0; j < CH; ++j) f[k][j] = pi_ld16(fc1 + (size_t)(wave * OWN + b * HELD + k) * COLS + j * 512 + lane * 8);
    };
    fetch1(f1[0], 0);
#pragma unroll
    for (int l = 0; l < NL; ++l) f2[l] = pi_ld16(fc2 + (size_t)(n0 + wave * 8 + l * NPL + lane / LPN) * R + lane % LPN * 8);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        if (KIND >= 1) fetch8(wv[j], nw + j * 512 + lane * 8);
        if (KIND == 2) fetch8(bv[j], nb + j * 512 + lane * 8);
    }
    auto packed = [](const float (&v)[8]) {
        const __half2 h[4] = {__floats2half2_rn(v[0], v[1]), __floats2half2_rn(v[2], v[3]), __floats2half2_rn(v[4], v[5]), __floats2half2_rn(v[6], v[7])};
        return *reinterpret_cast<const pi_u32x4 *>(h);
    };
    if constexpr (SUM) {
        for (int s0 = 0; s0 < n_shares; s0 += kSmShares) {
            if (s0) fetch_shares(s0);
#pragma unroll
            for (int s = 0; s < kSmShares; ++s)
                if (s0 + s < n_shares)
#pragma unroll
                    for (int j = 0; j < CH; ++j)
#pragma unroll
                        for (int k = 0; k < 8; ++k) xv[j][k] += sv[s][j][k];
        }
        if (blockIdx.x == 0 && wave == 0)
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                float * p = xsum + j * 512 + lane * 8;
                *reinterpret_cast<float4 *>(p) = make_float4(xv[j][0], xv[j][1], xv[j][2], xv[j][3]);
                *reinterpret_cast<float4 *>(p + 4) = make_float4(xv[j][4], xv[j][5], xv[j][6], xv[j][7]);
            }
    }
    pi_u32x4 xr[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) xr[j] = packed(xv[j]);
    // ---- hidden units: R / 4 a wave, HELD of them at a time ----
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b + 1 < NB) fetch1(f1[(b + 1) & 1], b + 1);
#pragma unroll
        for (int k = 0; k < HELD; ++k) {
            float d = 0.0f;
#pragma unroll
            for (int j = 0; j < CH; ++j) d = pi_dot8h(f1[b & 1][k][j], xr[j], d);
            d = pi_wave_sum(d);
            if (lane == 0) hid[wave * OWN + b * HELD + k] = __float2half_rn(fmaxf(d, 0.0f));
        }
    }
    // ---- the FFN's input (its values in place of x's) ----
    if (KIND >= 1) {
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) s += KIND == 1 ? (double)__fmul_rn(xv[j][k], xv[j][k]) : (double)xv[j][k];
        s = pi_wave_sum_f64(s);
        float mean = 0.0f;
        if (KIND == 2) {
            mean = (float)(s / COLS);
            s = 0.0;
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int k = 0; k < 8; ++k) { const float v = __fsub_rn(xv[j][k], mean); s += (double)__fmul_rn(v, v); }
            s = pi_wave_sum_f64(s);
        }
        const float scale = pi_inv_sqrt((float)(s / COLS) + eps);
#pragma unroll
        for (int j = 0; j < CH; ++j) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float v = __fmul_rn(__fmul_rn(KIND == 2 ? __fsub_rn(xv[j][k], mean) : xv[j][k], scale), wv[j][k]);
                if (KIND == 2) v = __fadd_rn(v, bv[j][k]);
                xv[j][k] = v;
            }
            xr[j] = packed(xv[j]);
        }
    }
    __syncthreads();
    // ---- logits: LPN lanes a neuron, the sums in the order of a whole wave's ----
    {
        const pi_u32x4 h = *reinterpret_cast<const pi_u32x4 *>(hid + lane % LPN * 8);
        uint32_t mine = 0;
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            float d = pi_dot8h(f2[l], h, 0.0f);
            d += pi_dpp_f32<PI_DPP_XOR1, 0xF>(d);
            d += pi_dpp_f32<PI_DPP_XOR2, 0xF>(d);
            d += pi_dpp_f32<PI_DPP_HALF_MIRROR, 0xF>(d);
            if (LPN >= 16) d += pi_dpp_f32<PI_DPP_MIRROR, 0xF>(d);
            if (LPN == 32) d += pi_dpp_f32<PI_DPP_BCAST15, 0xA>(d);               // (whole in the second half of each 32 lanes)
            const unsigned long long on = __ballot(!(d < thr));
#pragma unroll
            for (int k = 0; k < NPL; ++k) mine |= (uint32_t)(on >> (k * LPN + (LPN == 32 ? 16 : 0)) & 1) << (l * NPL + k);
        }
        if (lane == 0) word[wave] = mine << (8 * wave);
    }
    __syncthreads();
    uint32_t all = __builtin_amdgcn_readfirstlane(word[0] | word[1] | word[2] | word[3]);
    if (tid == 0) words[blockIdx.x] = all;
    // ---- rows: the active neurons number wave, wave + 4, .. are this wave's ----
    float acc[CH][8];
#pragma unroll
    for (int j = 0; j < CH; ++j)
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[j][k] = 0.0f;
    for (int k = 0; k < wave && all; ++k) all &= all - 1;
    while (all) {
        int n[kSmAtOnce], live = 0;
#pragma unroll
        for (int u = 0; u < kSmAtOnce; ++u) {                       // (past the last one its rows again, under a weight of zero)
            n[u] = all ? __builtin_ctz(all) : n[u ? u - 1 : 0];
            if (all) ++live;
#pragma unroll
            for (int k = 0; k < 4; ++k) all &= all - 1;             // (0 stays 0)
        }
        pi_u32x4 ru[kSmAtOnce][CH], rg[kSmAtOnce][CH], rd[kSmAtOnce][CH];
#pragma unroll
        for (int u = 0; u < kSmAtOnce; ++u)
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const size_t at = (size_t)(n0 + n[u]) * COLS + j * 512 + lane * 8;
                ru[u][j] = pi_ld16(up + at);
                if (GATE) rg[u][j] = pi_ld16(gate + at);
                rd[u][j] = pi_ld16(down + at);
            }
#pragma unroll
        for (int u = 0; u < kSmAtOnce; ++u) {
            if (u >= live) break;
            float a = 0.0f, b = 0.0f;
#pragma unroll
            for (int j = 0; j < CH; ++j) { a = pi_dot8h(ru[u][j], xr[j], a); if (GATE) b = pi_dot8h(rg[u][j], xr[j], b); }
            a = pi_wave_sum(a);
            if (GATE) b = pi_wave_sum(b);
            const float h = pi_round_f16(GATE ? __fmul_rn(fmaxf(b, 0.0f), a) : fmaxf(a, 0.0f));
            if (h == 0.0f) continue;                                // (no term, as on the CPU path: a zero times an infinite weight would be one)
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                float f[8];
                pi_unpack8(rd[u][j], f);
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[j][k] = fmaf(f[k], h, acc[j][k]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        float * p = &part[wave][j * 512 + lane * 8];
        *reinterpret_cast<float4 *>(p) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
        *reinterpret_cast<float4 *>(p + 4) = make_float4(acc[j][4], acc[j][5], acc[j][6], acc[j][7]);
    }
    __syncthreads();
    for (int c = tid; c < COLS; c += kSmBlock) partial[(size_t)blockIdx.x * COLS + c] = ((part[0][c] + part[1][c]) + part[2][c]) + part[3][c];
}

}  // namespace

static int ffn_small(const float * shares, int n_shares, float * xsum, const void * fc1_f16, const void * fc2_f16, int ff, int r, float threshold, const void * up_f16, const void * gate_f16, const void * down_t_f16, int cols, const float * x,
                          const pi_norm * norm, int epilogue, const float * add1, const float * add2, float * out, int32_t * n_active, pi_workspace * ws, pi_stream_t stream) {
    if (!fc1_f16 || !fc2_f16 || !up_f16 || !down_t_f16 || !x || !out || !ws) return pi::fail(PI_E_ARG, "pi_k_sparse_ffn_small: null pointer");
    const NormArgs na{norm ? norm->kind : 0, norm ? norm->eps : 0.0f, norm ? norm->w : nullptr, norm ? norm->b : nullptr};
    if (!pi_k_sparse_ffn_small_supported(ff, r, cols) || !(na.kind == 0 || (na.kind == 1 && na.w && !na.b) || (na.kind == 2 && na.w && na.b)))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_sparse_ffn_small: 512 or 1024 columns, rank 64, 128 or 256, predictor of at most 131072 values, ff % 32 == 0, a norm with its weights");
    if (ff > ws->max_ff || cols > ws->max_d) return pi::fail(PI_E_ARG, "pi_k_sparse_ffn_small: shape exceeds the workspace");
    if ((((uintptr_t)fc1_f16 | (uintptr_t)fc2_f16 | (uintptr_t)up_f16 | (uintptr_t)gate_f16 | (uintptr_t)down_t_f16 | (uintptr_t)x | (uintptr_t)na.w | (uintptr_t)na.b) & 15) != 0)
        return pi::fail(PI_E_ARG, "pi_k_sparse_ffn_small: operands must be 16-byte aligned");
    const __half * a = (const __half *)fc1_f16, * b = (const __half *)fc2_f16, * u = (const __half *)up_f16, * g = (const __half *)gate_f16, * d = (const __half *)down_t_f16;
#define PI_SM(CH, R, GATE, KIND, SUM) hipLaunchKernelGGL((ffn_small_f16_kernel<CH, R, GATE, KIND, SUM>), dim3(ff / kSmNeurons), dim3(kSmBlock), 0, (hipStream_t)stream, a, b, u, g, d, x, na.w, na.b, na.eps, threshold, ws->words, ws->ffn_partial, shares, n_shares, xsum)
#define PI_SM_K(CH, R, GATE) do { if (na.kind == 0) PI_SM(CH, R, GATE, 0, false); else if (na.kind == 1) PI_SM(CH, R, GATE, 1, false); else PI_SM(CH, R, GATE, 2, false); } while (0)
#define PI_SM_G(CH, R) do { if (shares) PI_SM(CH, R, true, 1, true); else if (g) PI_SM_K(CH, R, true); else PI_SM_K(CH, R, false); } while (0)
    if (cols == 512) { if (r == 64) PI_SM_G(1, 64); else if (r == 128) PI_SM_G(1, 128); else PI_SM_G(1, 256); }
    else             { if (r == 64) PI_SM_G(2, 64); else PI_SM_G(2, 128); }
#undef PI_SM_G
#undef PI_SM_K
#undef PI_SM
    ws->pf_parts = ws->pf_words = ff / kSmNeurons;
    const int rc = pi::check_launch("pi_k_sparse_ffn_small");
    return rc != PI_OK ? rc : pi_k_sparse_ffn_reduce(ff, cols, epilogue, add1, add2, out, n_active, ws, stream);
}

namespace pi {
int sparse_ffn_small_of(const float * parts, int n_parts, float * xsum, const void * fc1_f16, const void * fc2_f16, int ff, int r, float threshold, const void * up_f16, const void * gate_f16,
                        const void * down_t_f16, int cols, const float * x, const pi_norm * norm, float * out, int32_t * n_active, pi_workspace * ws, pi_stream_t stream) {
    if (!parts || n_parts <= 0 || n_parts > kOutHeads || !xsum || !gate_f16 || !norm || norm->kind != 1 || (((uintptr_t)parts | (uintptr_t)xsum) & 15)) return fail(PI_E_ARG, "sparse_ffn_small_of: bad arguments");
    return ffn_small(parts, n_parts, xsum, fc1_f16, fc2_f16, ff, r, threshold, up_f16, gate_f16, down_t_f16, cols, x, norm, PI_EPI_ADD, xsum, nullptr, out, n_active, ws, stream);
}
}  // namespace pi

extern "C" {

// A first predictor matrix of 256 KB at most.  Against the four launches, with a tenth (half) of the neurons active, us: 512 columns, rank 64, 1024 neurons
// 7.8 : 16.1 (8.4 : 17.4), 32768 13.3 : 37.2 (17.3 : 112); rank 256, 1024 neurons 14.0 : 16.4, 16384 19.2 : 22.3 (21.4 : 61); 1024 columns, rank 128,
// 1024 neurons 11.3 : 17.4, 32768 27.4 : 38.7 (35.4 : 116).  Twice that matrix would be 9 us more in every one.
int pi_k_sparse_ffn_small_supported(int ff, int r, int cols) {
    return (cols == 512 || cols == 1024) && (r == 64 || r == 128 || r == 256) && r * cols <= 128 * 1024 && ff > 0 && ff % kSmNeurons == 0 && ff <= 32768;
}

int pi_k_sparse_ffn_small(const void * fc1_f16, const void * fc2_f16, int ff, int r, float threshold, const void * up_f16, const void * gate_f16, const void * down_t_f16, int cols, const float * x,
                          const pi_norm * norm, int epilogue, const float * add1, const float * add2, float * out, int32_t * n_active, pi_workspace * ws, pi_stream_t stream) {
    return ffn_small(nullptr, 0, nullptr, fc1_f16, fc2_f16, ff, r, threshold, up_f16, gate_f16, down_t_f16, cols, x, norm, epilogue, add1, add2, out, n_active, ws, stream);
}

}  // extern "C"
