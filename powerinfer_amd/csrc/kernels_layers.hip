// Operators of the models that are described layer by layer, apart from attention: embedding + norm, the pair of norms of a parallel
// layer, grouped mat-muls (heads of a latent attention, experts), rotation angles, expert choice, and the sum that closes a layer.
// Templated on the storage of activations: bf16 (matrix cores on bf16 operands, fp32 accumulation) or fp32.
#include "gemm_wide.hpp"
#include "layer_types.hpp"
#include "mixers.hpp"
#include "route.hpp"

namespace {

// ---------------------------------------------------------------------------------------------------------------------------------
// norms
// ---------------------------------------------------------------------------------------------------------------------------------
// 1 / sqrt(mean(x^2) + eps) of a row the workgroup reads together (squares summed in fp64, fixed order)
template <typename LD> __device__ float row_rms_scale(int cols, float eps, double * red, LD && ld) {
    double s = 0.0;
    for (int i = threadIdx.x; i < cols; i += blockDim.x) { const float v = ld(i); s += (double)v * (double)v; }
    s = block_sum_f64(s, red);
    return pi_inv_sqrt((float)(s / cols) + eps);
}

// eight columns a thread at a time, up to 8192 of them in the registers of 256 threads (rows on 16 bytes): a value a thread, 2 bytes of a row and 1024 threads took
// 2048 tokens of 4096 columns 32 us, this 12; narrow rows have fewer waves (2048 tokens of 512 columns 4.7, 4.9 with 256 threads, 3.4 with 64)
__device__ void embed_norm_row(const uint16_t * __restrict__ row, int cols, const float * __restrict__ w, float eps, float * __restrict__ out, double * red) {
    constexpr int N = 4;
    if (cols % 8 == 0 && cols <= N * 8 * (int)blockDim.x && (((uintptr_t)row | (uintptr_t)w | (uintptr_t)out) & 15) == 0) {
        pi_u32x4 r[N];
        float4 wv[N][2];
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int i = ((int)threadIdx.x + k * (int)blockDim.x) * 8;
            r[k] = pi_u32x4{0, 0, 0, 0};
            if (i < cols) { r[k] = pi_ld16(row + i); wv[k][0] = *reinterpret_cast<const float4 *>(w + i); wv[k][1] = *reinterpret_cast<const float4 *>(w + i + 4); }
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float lo = __uint_as_float(r[k][j] << 16), hi = __uint_as_float(r[k][j] & 0xffff0000u);
                s += (double)lo * (double)lo + (double)hi * (double)hi;
            }
        s = block_sum_f64(s, red);
        const float sc = pi_inv_sqrt((float)(s / cols) + eps);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int i = ((int)threadIdx.x + k * (int)blockDim.x) * 8;
            if (i >= cols) break;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4 g = wv[k][h];
                const float v[4] = {__uint_as_float(r[k][2 * h] << 16), __uint_as_float(r[k][2 * h] & 0xffff0000u), __uint_as_float(r[k][2 * h + 1] << 16), __uint_as_float(r[k][2 * h + 1] & 0xffff0000u)};
                *reinterpret_cast<float4 *>(out + i + 4 * h) = make_float4(v[0] * sc * g.x, v[1] * sc * g.y, v[2] * sc * g.z, v[3] * sc * g.w);
            }
        }
        return;
    }
    const float sc = row_rms_scale(cols, eps, red, [&](int i) { return bf16_to_f32(row[i]); });
    for (int i = threadIdx.x; i < cols; i += blockDim.x) out[i] = bf16_to_f32(row[i]) * sc * w[i];
}
inline int embed_norm_block(int cols) { return cols % 8 == 0 && cols <= 8192 ? std::max(64, std::min((cols + 511) / 512 * 64, 256)) : cols > 2048 ? 1024 : 256; }
__global__ __launch_bounds__(1024) void embed_norm_kernel(const uint16_t * __restrict__ table, int cols, const int32_t * __restrict__ tokens,
                                                          const float * __restrict__ w, float eps, float * __restrict__ x) {
    __shared__ double red[16];
    embed_norm_row(table + (size_t)tokens[blockIdx.x] * cols, cols, w, eps, x + (size_t)blockIdx.x * cols, red);
}

template <typename ST>
__global__ __launch_bounds__(1024) void norm_pair_kernel(const float * __restrict__ x, const int32_t * __restrict__ rows, int cols, float eps,
                                                        const float * __restrict__ wa, ST * __restrict__ out_a, const float * __restrict__ wb,
                                                        ST * __restrict__ out_b, int ld, int ol) {
    __shared__ double red[16];
    const float * xt = x + (size_t)(rows ? rows[blockIdx.x] : blockIdx.x) * cols;
    auto at = [&](int i) -> size_t { return ol ? pi_ol_index(blockIdx.x, i) : (size_t)blockIdx.x * ld + i; };
    if (cols <= 4 * (int)blockDim.x) {              // one memory round trip: the row and both weight vectors are requested together
        float xv[4], av[4], bv[4];
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            xv[k] = i < cols ? xt[i] : 0.0f;
            av[k] = i < cols ? wa[i] : 0.0f;
            bv[k] = wb && i < cols ? wb[i] : 0.0f;
            s += (double)xv[k] * (double)xv[k];
        }
        s = block_sum_f64(s, red);
        const float sc = pi_inv_sqrt((float)(s / cols) + eps);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            if (i < cols) {
                out_a[at(i)] = to_st<ST>(xv[k] * sc * av[k]);
                if (wb) out_b[at(i)] = to_st<ST>(xv[k] * sc * bv[k]);
            }
        }
        return;
    }
    const float sc = row_rms_scale(cols, eps, red, [&](int i) { return xt[i]; });
    for (int i = threadIdx.x; i < cols; i += blockDim.x) {
        const float v = xt[i] * sc;
        out_a[at(i)] = to_st<ST>(v * wa[i]);
        if (wb) out_b[at(i)] = to_st<ST>(v * wb[i]);
    }
}

// the same with four columns a thread at a time, up to 4096 of them in the registers of 256 threads (rows, weights and outputs in whole quads): 2048 tokens of 4096
// columns into two operands 22.8 -> 12.6 us.  For long passes: 16 waves a row are the better ones for a few (one token 4.8 us, this 5.1); and beyond 512 columns,
// below which most threads have none (2048 tokens of 512 columns 4.5 us, this 5.4; of 768 7.4 and 5.8)
template <typename ST>
__global__ __launch_bounds__(256) void norm_pair_quads_kernel(const float * __restrict__ x, const int32_t * __restrict__ rows, int cols, float eps, const float * __restrict__ wa,
                                                             ST * __restrict__ out_a, const float * __restrict__ wb, ST * __restrict__ out_b, int ld) {
    constexpr int N = 4;
    __shared__ double red[4];
    const float * xt = x + (size_t)(rows ? rows[blockIdx.x] : blockIdx.x) * cols;
    float4 xv[N], av[N], bv[N];
    const int last = cols - 4;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int i = min(((int)threadIdx.x + k * 256) * 4, last);
        xv[k] = *reinterpret_cast<const float4 *>(xt + i);
        av[k] = *reinterpret_cast<const float4 *>(wa + i);
        if (wb) bv[k] = *reinterpret_cast<const float4 *>(wb + i);
    }
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < N; ++k)
        if (((int)threadIdx.x + k * 256) * 4 < cols) s += ((double)xv[k].x * (double)xv[k].x + (double)xv[k].y * (double)xv[k].y) + ((double)xv[k].z * (double)xv[k].z + (double)xv[k].w * (double)xv[k].w);
    s = block_sum_f64(s, red);
    const float sc = pi_inv_sqrt((float)(s / cols) + eps);
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int i = ((int)threadIdx.x + k * 256) * 4;
        if (i >= cols) break;
        const size_t at = (size_t)blockIdx.x * ld + i;
        const float a[4] = {xv[k].x * sc * av[k].x, xv[k].y * sc * av[k].y, xv[k].z * sc * av[k].z, xv[k].w * sc * av[k].w};
        store4(out_a + at, a, true, 4);
        if (wb) {
            const float b[4] = {xv[k].x * sc * bv[k].x, xv[k].y * sc * bv[k].y, xv[k].z * sc * bv[k].z, xv[k].w * sc * bv[k].w};
            store4(out_b + at, b, true, 4);
        }
    }
}

struct Bigram { const uint16_t * table; float scale; const uint16_t * bigram; int buckets; long long mul_prev, mul_cur; };
__device__ void embed_bigram_row(const Bigram & g, int cols, int tok, int before, float * __restrict__ o, float * __restrict__ o0) {
    const uint16_t * a = g.table + (size_t)tok * cols, * b = nullptr;
    if (g.bigram) b = g.bigram + (size_t)(before < 0 ? g.buckets : (int)(((long long)before * g.mul_prev + (long long)tok * g.mul_cur) % g.buckets)) * cols;
    if ((cols & 7) == 0) {
        for (int i = threadIdx.x * 8; i < cols; i += blockDim.x * 8) {
            const pi_u32x4 u = pi_ld16(a + i), w = b ? pi_ld16(b + i) : pi_u32x4{0, 0, 0, 0};
            float v[8];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[2 * j] = __uint_as_float(u[j] << 16) * g.scale + __uint_as_float(w[j] << 16);
                v[2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u) * g.scale + __uint_as_float(w[j] & 0xffff0000u);
            }
#pragma unroll
            for (int j = 0; j < 8; j += 4) {
                *reinterpret_cast<float4 *>(o + i + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
                if (o0) *reinterpret_cast<float4 *>(o0 + i + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
            }
        }
    } else {
        for (int i = threadIdx.x; i < cols; i += blockDim.x) {
            const float v = bf16_to_f32(a[i]) * g.scale + (b ? bf16_to_f32(b[i]) : 0.0f);
            o[i] = v;
            if (o0) o0[i] = v;
        }
    }
}
__global__ __launch_bounds__(256) void embed_bigram_kernel(Bigram g, int cols, const int32_t * __restrict__ tokens, int32_t * prev, int carry, float * __restrict__ x, float * __restrict__ x0) {
    const int t = blockIdx.x, tok = tokens[t];
    embed_bigram_row(g, cols, tok, prev[t], x + (size_t)t * cols, x0 ? x0 + (size_t)t * cols : nullptr);
    if (carry) {
        __syncthreads();                               // every thread has read prev[t]
        if (threadIdx.x == 0) prev[t] = tok;
    }
}

// layer norm, two passes over the row (held in registers where it fits); x0, step: added to the residual stream first
template <typename ST>
__global__ __launch_bounds__(1024) void layer_norm_kernel(float * __restrict__ x, const int32_t * __restrict__ rows, int cols, float eps, const float * __restrict__ w,
                                                         const float * __restrict__ x0, const float * __restrict__ step, ST * __restrict__ out, int ld, int ol) {
    __shared__ double red[16];
    const size_t base = (size_t)(rows ? rows[blockIdx.x] : blockIdx.x) * cols;
    float * xt = x + base;
    auto at = [&](int i) -> size_t { return ol ? pi_ol_index(blockIdx.x, i) : (size_t)blockIdx.x * ld + i; };
    const bool adds = x0 || step;
    if (cols <= 4 * (int)blockDim.x) {
        float xv[4], wv[4];
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            xv[k] = i < cols ? xt[i] : 0.0f;
            wv[k] = i < cols ? w[i] : 0.0f;
            if (x0 && i < cols) xv[k] += x0[base + i];
            if (step && i < cols) xv[k] += step[i];
            s += (double)xv[k];
        }
        const float mean = (float)(block_sum_f64(s, red) / cols);
        s = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            if (i < cols) {
                if (adds) xt[i] = xv[k];
                xv[k] -= mean;
                s += (double)xv[k] * (double)xv[k];
            }
        }
        const float sc = pi_inv_sqrt((float)(block_sum_f64(s, red) / cols) + eps);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            if (i < cols) out[at(i)] = to_st<ST>(xv[k] * sc * wv[k]);
        }
        return;
    }
    double s = 0.0;
    for (int i = threadIdx.x; i < cols; i += blockDim.x) {
        float v = xt[i];
        if (x0) v += x0[base + i];
        if (step) v += step[i];
        if (adds) xt[i] = v;                           // (read back below by the thread that wrote it)
        s += (double)v;
    }
    const float mean = (float)(block_sum_f64(s, red) / cols);
    s = 0.0;
    for (int i = threadIdx.x; i < cols; i += blockDim.x) { const float v = xt[i] - mean; s += (double)v * (double)v; }
    const float sc = pi_inv_sqrt((float)(block_sum_f64(s, red) / cols) + eps);
    for (int i = threadIdx.x; i < cols; i += blockDim.x) out[at(i)] = to_st<ST>((xt[i] - mean) * sc * w[i]);
}

// what closes a sublayer whose norm comes after the sum (pi_res_norm): Q quads of columns per thread in registers, one trip over the row
template <typename ST, int Q>
__global__ void res_norm_kernel(pi_res_norm p) {
    __shared__ double red[16];
    const int t = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const size_t base = (size_t)t * p.cols;
    const float * gz = p.gate_z ? p.gate_z + (size_t)t * p.ld_gate + p.off_gate : nullptr;
    float v[Q][4], wv[Q][4];
    double s = 0.0;
    const bool quads = ((p.cols | p.ld_gate | p.off_gate) & 3) == 0;
    auto load = [&](const float * a, int c, float (&o)[4]) {      // columns c .. c + 3 of a row (past its end: zeros)
        if (quads && c < p.cols) { const float4 q = *reinterpret_cast<const float4 *>(a + c); o[0] = q.x; o[1] = q.y; o[2] = q.z; o[3] = q.w; }
        else for (int j = 0; j < 4; ++j) o[j] = c + j < p.cols ? a[c + j] : 0.0f;
    };
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = (tid + q * nt) * 4;
        load(p.x + base, c, v[q]);
        if (p.w) load(p.w, c, wv[q]);
        if (p.mix) {
            float m[4];
            load(p.mix + base, c, m);
            if (gz) {
                float g[4], b[4];
                load(gz, c, g);
                load(p.gate_b, c, b);
#pragma unroll
                for (int j = 0; j < 4; ++j) m[j] *= sigmoid_f32(g[j] + b[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) v[q][j] = fmaf(p.alpha, v[q][j], m[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) if (c + j < p.cols) s += (double)v[q][j] * (double)v[q][j];
    }
    float sc = 1.0f;
    if (p.w) sc = pi_inv_sqrt((float)(block_sum_f64(s, red) / p.cols) + p.eps);
    ST * h = (ST *)p.h;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int c = (tid + q * nt) * 4;
        if (c >= p.cols) break;
        if (p.w) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[q][j] *= sc * wv[q][j];
        }
        const bool whole = quads && c + 4 <= p.cols;
        store4(p.out + base + c, v[q], whole, p.cols - c);
        if (p.keep) store4(p.keep + base + c, v[q], whole, p.cols - c);
        if (h) {                                       // (four columns from a multiple of four on lie together in both layouts)
            ST * o = h + (p.ol ? pi_ol_index(t, c) : (size_t)t * p.ld + c);
            store4(o, v[q], ((uintptr_t)o & (4 * sizeof(ST) - 1)) == 0 && c + 4 <= p.cols, p.cols - c);
        }
    }
}
template <typename ST> int launch_res_norm(const pi_res_norm & p, hipStream_t st) {
    const int quads = (p.cols + 3) / 4;
    if (quads <= 256) hipLaunchKernelGGL((res_norm_kernel<ST, 1>), dim3(p.T), dim3(256), 0, st, p);
    else if (quads <= 512) hipLaunchKernelGGL((res_norm_kernel<ST, 1>), dim3(p.T), dim3(512), 0, st, p);
    else if (quads <= 1024) hipLaunchKernelGGL((res_norm_kernel<ST, 2>), dim3(p.T), dim3(512), 0, st, p);
    else if (quads <= 2048) hipLaunchKernelGGL((res_norm_kernel<ST, 4>), dim3(p.T), dim3(512), 0, st, p);
    else if (quads <= 8192) hipLaunchKernelGGL((res_norm_kernel<ST, 8>), dim3(p.T), dim3(1024), 0, st, p);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_res_norm: up to 32768 columns");
    return pi::check_launch("pi_k_res_norm");
}

template <typename ST>
__global__ __launch_bounds__(256) void ffn_front_kernel(pi_ffn_front f, const float * __restrict__ z, int ldz, int per) {
    extern __shared__ __align__(16) float sm[];
    front_block<ST>(f, z, ldz, blockIdx.x / per, blockIdx.x % per, sm);
}

// ---------------------------------------------------------------------------------------------------------------------------------
// grouped mat-mul.  A workgroup of four waves owns 64 rows of one group's matrix x 32 of the group's tokens; each wave holds 16 rows in
// the matrix cores' operand layout (lane l: row l % 16, eight consecutive columns 8 * (l / 16) of a 32-column step) against two token
// tiles.  fp32 storage runs the same steps on v_mfma_f32_16x16x4_f32, eight per 32 columns.
// ---------------------------------------------------------------------------------------------------------------------------------
template <typename ST>
__global__ __launch_bounds__(256) void group_gemm_kernel(pi_group_gemm g) {
    const int grp = blockIdx.z;
    const int lo = g.off ? g.off[grp] : 0, n = g.off ? g.off[grp + 1] - lo : g.T;
    const int t0 = blockIdx.y * 32;
    if (t0 >= n) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const int row0 = blockIdx.x * 64 + wave * 16;
    if (row0 >= g.rows) return;
    const uint16_t * W = (const uint16_t *)g.W + (size_t)grp * g.w_gs + (size_t)min(row0 + i, g.rows - 1) * g.ldw + q * 8;
    const ST * xb = (const ST *)g.x + (g.off ? 0 : (size_t)grp * g.x_gs);
    const ST * xp[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int t = min(t0 + u * 16 + i, n - 1);
        const int xr = g.off ? (g.gather ? g.gather[lo + t] / g.gather_div : lo + t) : t;
        xp[u] = xb + (size_t)xr * g.ldx + q * 8;
    }
    pi_f4 acc[2] = {pi_f4{0, 0, 0, 0}, pi_f4{0, 0, 0, 0}};
    const bool two = t0 + 16 < n;
    for (int k = 0; k < g.cols; k += 32) {
        const Frag<ST> a = frag_weights<ST>(W + k);
        frag_mma(a, frag_load(xp[0] + k), acc[0]);
        if (two) frag_mma(a, frag_load(xp[1] + k), acc[1]);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int t = t0 + u * 16 + i;
        if (t >= n) continue;
        const float alpha = g.pair_w ? g.alpha * g.pair_w[g.gather[lo + t]] : g.alpha, one = g.glu_plain_up ? 0.0f : 1.0f;
        const size_t yr = g.off ? (size_t)(lo + t) * g.ldy : (size_t)grp * g.y_gs + (size_t)t * g.ldy;
        if (g.glu) {                                   // rows in (gate, up) pairs: a lane holds two of them
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const int row = row0 + 4 * q + r;
                if (row >= g.rows) continue;
                const float v = clamped_glu(acc[u][r] * alpha, acc[u][r + 1] * alpha, g.glu_limit, g.glu_gain, one);
                if (g.y_f32) ((float *)g.y)[yr + row / 2] = v;
                else ((ST *)g.y)[yr + row / 2] = to_st<ST>(v);
            }
            continue;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + 4 * q + r;
            if (row >= g.rows) continue;
            float v = acc[u][r] * alpha;
            if (g.relu2) { v = fmaxf(v, 0.0f); v *= v; }
            if (g.y_f32) ((float *)g.y)[yr + row] = v;
            else ((ST *)g.y)[yr + row] = to_st<ST>(v);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// rotation angles: formed and reduced in fp64, so that the fp32 cosine and sine are right at any position
// ---------------------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ float2 rope_angle_at(int pos, int i, int dims, double base, const double * freq, double length) {
    double s, c;
    sincos((double)pos * (freq ? freq[i] : pow(base, -2.0 * (double)i / (double)dims)), &s, &c);
    return freq ? make_float2((float)(length * c), (float)(length * s)) : make_float2((float)c, (float)s);
}
__global__ void rope_angles_kernel(const int32_t * __restrict__ pos, int T, int dims, double base, float2 * __restrict__ cs) {
    const int half = dims / 2, idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < T * half) cs[idx] = rope_angle_at(pos[idx / half], idx % half, dims, base, nullptr, 1.0);
}

__global__ void rope_table_kernel(const int32_t * __restrict__ pos, int T, int half, const double * __restrict__ freq, double length, float2 * __restrict__ cs) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < T * half) cs[idx] = rope_angle_at(pos[idx / half], idx % half, 2 * half, 0.0, freq, length);
}

// What a pass begins with, in one launch: its integers on their way from pinned memory to the device, the new cells into their sequences' lists, the
// embeddings and the rotations' angles.  A copy and up to four launches were 11 us on the device and more for the host to issue, with nothing
// to run beside them.  A short pass reads its tokens and positions in pinned memory as well; a long one is two launches, as each such read
// crosses the link: the copy, then the rest from device memory.
__global__ __launch_bounds__(1024) void pass_start_kernel(pi::PassStart p, Bigram g, int embeds, int copies, int appends) {
    __shared__ double red[16];
    const int tid = threadIdx.x, nt = blockDim.x;
    int b = blockIdx.x;
    if (b < embeds) {
        const int tok = p.tokens[b];
        float * x = p.x + (size_t)b * p.cols;
        if (p.norm) embed_norm_row((const uint16_t *)p.table + (size_t)tok * p.cols, p.cols, p.norm, p.eps, x, red);
        else embed_bigram_row(g, p.cols, tok, p.prev[b], x, p.x0 ? p.x0 + (size_t)b * p.cols : nullptr);
        return;
    }
    b -= embeds;
    if (b < copies) {                                  // (both sides start on 16 bytes)
        const size_t i = ((size_t)b * nt + tid) * 4;
        if (i + 4 <= p.words) *reinterpret_cast<int4 *>(p.dst + i) = *reinterpret_cast<const int4 *>(p.src + i);
        else for (size_t k = i; k < p.words; ++k) p.dst[k] = p.src[k];
        return;
    }
    b -= copies;
    if (b < appends) {
        const int i = b * nt + tid;
        if (i < p.n_append) p.lists[(size_t)p.append[3 * i] * p.list_ld + p.append[3 * i + 1]] = p.append[3 * i + 2];
        return;
    }
    b -= appends;
    for (int k = 0; k < p.n_rot; ++k) {
        const pi::PassStart::Rot & r = p.rot[k];
        const int half = r.dims / 2, n = (p.T * half + nt - 1) / nt, idx = b * nt + tid;
        if (b < n) {
            if (idx < p.T * half) reinterpret_cast<float2 *>(r.cs)[idx] = rope_angle_at(p.pos[idx / half], idx % half, r.dims, r.base, r.freq, r.length);
            return;
        }
        b -= n;
    }
}

// The router's products of a long pass: 64 tokens and 512 columns a workgroup, whose sums go apart to the choice behind them, which adds them up.  As tiles of 64 rows
// and 64 tokens over all columns they were one row of tiles, all on one of the eight XCDs, each reading 1 MB: 2048 tokens of 4096 columns, 64 experts
// 25.3 -> 10.3 us (and 1.6 more for the choice).  Bound by the 128 KB that a unit reads: the experts' columns go through LDS (read by each wave for itself 15.4 us), a wave holds its 16
// tokens' values.
constexpr int kRouterCols = 512, kRouterExperts = 128, kRouterPitch = kRouterCols * 2 + 16;      // (16 bytes on: sixteen rows' pieces in different banks)
__global__ __launch_bounds__(256) void router_parts_kernel(const bf16 * __restrict__ W, int E, int cols, const bf16 * __restrict__ x, int T, float * __restrict__ parts) {
    extern __shared__ __align__(16) unsigned char smem[];           // [E rounded up to 16][kRouterPitch]
    constexpr int N = kRouterCols / 32, ROWS = 16;                  // rows a wave requests together
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4, k0 = (int)blockIdx.y * kRouterCols, tok = (int)blockIdx.x * 64 + wave * 16 + i;
    const int n_m = (E + 15) / 16;
    pi_u32x4 b[N], w[ROWS];
    const bf16 * xt = x + (size_t)min(tok, T - 1) * cols + k0 + g * 8;
    for (int r0 = wave; r0 < n_m * 16; r0 += 4 * ROWS) {
#pragma unroll
        for (int k = 0; k < ROWS; ++k) w[k] = pi_ld16(W + (size_t)min(r0 + 4 * k, E - 1) * cols + k0 + lane * 8);
        if (r0 == wave) {
#pragma unroll
            for (int k = 0; k < N; ++k) b[k] = pi_ld16(xt + k * 32);
        }
#pragma unroll
        for (int k = 0; k < ROWS; ++k)
            if (r0 + 4 * k < n_m * 16) *reinterpret_cast<pi_u32x4 *>(smem + (size_t)(r0 + 4 * k) * kRouterPitch + lane * 16) = w[k];
    }
    __syncthreads();
    float * out = parts + ((size_t)blockIdx.y * T + tok) * E;
    for (int m = 0; m < n_m; ++m) {
        pi_f4 acc[2] = {};
        const unsigned char * p = smem + (size_t)(m * 16 + i) * kRouterPitch + g * 16;
#pragma unroll
        for (int k = 0; k < N; ++k) acc[k & 1] = mma16<__bf16>(*reinterpret_cast<const pi_u32x4 *>(p + k * 64), b[k], acc[k & 1]);
        if (tok >= T) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (m * 16 + 4 * g + r < E) out[m * 16 + 4 * g + r] = acc[0][r] + acc[1][r];
    }
}

// expert choice, one workgroup per token
__global__ __launch_bounds__(256) void route_kernel(RouteArgs r) {
    extern __shared__ __align__(16) float sm[];
    route_token(r, blockIdx.x, sm);
}

// Pairs in expert order, one workgroup with the experts' counters in LDS: counts, their prefix sums, places.  The order of the pairs
// within an expert is free (every row of the grouped products is computed on its own).  tiles (optional): {expert, first place} of
// every group of up to tile_n pairs of one expert, n_tiles of them - the token tiles of the grouped products.
__global__ __launch_bounds__(1024) void moe_sort_kernel(const int32_t * __restrict__ ids, int n, int E, int32_t * __restrict__ off, int32_t * __restrict__ perm,
                                                        int32_t * __restrict__ inv, int tile_n, int2 * __restrict__ tiles, int32_t * __restrict__ n_tiles) {
    extern __shared__ int cnt[];
    __shared__ int sred[16];
    for (int e = threadIdx.x; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < n; p += 1024) atomicAdd(&cnt[ids[p]], 1);
    __syncthreads();
    int base = 0, tbase = 0;
    for (int e0 = 0; e0 < E; e0 += 1024) {
        const int e = e0 + threadIdx.x, c = e < E ? cnt[e] : 0;
        int tot, ttot;
        const int at = base + block_exclusive_scan_i32(c, &tot, sred);
        const int nt = tiles ? (c + tile_n - 1) / tile_n : 0;
        const int ta = tbase + block_exclusive_scan_i32(nt, &ttot, sred);
        if (e < E) {
            off[e] = at;
            cnt[e] = at;
            for (int k = 0; k < nt; ++k) tiles[ta + k] = make_int2(e, at + k * tile_n);
        }
        base += tot; tbase += ttot;
    }
    if (threadIdx.x == 0) { off[E] = base; if (tiles) *n_tiles = tbase; }
    __syncthreads();
    for (int p = threadIdx.x; p < n; p += 1024) {
        const int at = atomicAdd(&cnt[ids[p]], 1);
        perm[at] = p;
        inv[p] = at;
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// grouped mat-mul of prompt portions (bf16): GemmTile per (group, token tile, row tile).  Token tiles come from moe_sort's list
// (g.tiles) or, without a list, every group has ceil(T / BN) of them.  The units are dealt out so that an XCD works through a
// contiguous range of them: the row tiles of a token tile, and the token tiles of a group, share that XCD's L2.
// ---------------------------------------------------------------------------------------------------------------------------------
// a wave's 16 x 16 tiles of outputs, rows from row0 and tokens from tok0 of the token tile (group grp, places lo .. lo + n - 1); lane = 16 q + i
template <int MT, int NT>
__device__ __forceinline__ void group_store(const pi_group_gemm & g, int grp, int lo, int n, int row0, int tok0, int q, int i, const pi_f4 (&acc)[MT][NT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int nn = 0; nn < NT; ++nn) {
            const int row = row0 + m * 16 + 4 * q, tok = tok0 + nn * 16 + i;
            if (tok >= n || row >= g.rows) continue;
            const float alpha = g.pair_w ? g.alpha * g.pair_w[g.gather[lo + tok]] : g.alpha;
            if (g.glu) {                               // rows in (gate, up) pairs: a lane holds two of them
                const size_t o = (g.off ? 0 : (size_t)grp * g.y_gs) + (size_t)(lo + tok) * g.ldy + row / 2;
                const float one = g.glu_plain_up ? 0.0f : 1.0f, a = clamped_glu(acc[m][nn][0] * alpha, acc[m][nn][1] * alpha, g.glu_limit, g.glu_gain, one);
                const float b = clamped_glu(acc[m][nn][2] * alpha, acc[m][nn][3] * alpha, g.glu_limit, g.glu_gain, one);
                const bool two = row + 4 <= g.rows;
                if (g.y_f32) {
                    ((float *)g.y)[o] = a;
                    if (two) ((float *)g.y)[o + 1] = b;
                } else if (two && (o & 1) == 0) {
                    const bf16 v[2] = {(bf16)a, (bf16)b};
                    *reinterpret_cast<uint32_t *>((bf16 *)g.y + o) = __builtin_bit_cast(uint32_t, v);
                } else {
                    ((bf16 *)g.y)[o] = (bf16)a;
                    if (two) ((bf16 *)g.y)[o + 1] = (bf16)b;
                }
                continue;
            }
            const size_t o = (g.off ? 0 : (size_t)grp * g.y_gs) + (size_t)(lo + tok) * g.ldy + row;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = acc[m][nn][r] * alpha;
                if (g.relu2) { v[r] = fmaxf(v[r], 0.0f); v[r] *= v[r]; }
            }
            const bool quad = row + 4 <= g.rows && (o & 3) == 0;
            if (g.y_f32) {
                float * y = (float *)g.y + o;
                if (quad) *reinterpret_cast<float4 *>(y) = make_float4(v[0], v[1], v[2], v[3]);
                else for (int r = 0; r < 4 && row + r < g.rows; ++r) y[r] = v[r];
            } else {
                bf16 * y = (bf16 *)g.y + o;
                bf16 b[4] = {(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
                if (quad) *reinterpret_cast<uint2 *>(y) = __builtin_bit_cast(uint2, b);
                else for (int r = 0; r < 4 && row + r < g.rows; ++r) y[r] = b[r];
            }
        }
}

// The column stage that the sums of these rows of a listed group begin with, in tiles of any size.  Rows a multiple of 4 KB apart lie in few of the memory's
// channels, and workgroups that began together would all read the same of them: 256 rows of a group have a place of their own there.  Tiles of 128
// and 256 tokens, us, one place for all / this: 64 experts of 96 tokens, 1408 x 4096 162 / 140, of 192 190 / 184; 8 experts of 64, 8192 x 4096 123 / 88, of
// 140 136 / 123; 1408 columns: no difference.  Tiles of 64 tokens gain nothing from it (16 experts of 33, 2816 x 2048: 36.1 / 36.5), but they keep the
// order of the larger ones.  The place goes by group and row alone, so that a token's outputs do not depend on how many come along.  Products without a list share
// their rows between many workgroups and begin at column 0 (every 2048 rows of 22016 x 5120 at another one: 400 tokens 1.5 % slower, 2043 tokens 3 % faster), as results in
// fp32 and short rows do.
__device__ __forceinline__ int group_first(const pi_group_gemm & g, int grp, int row0) {
    return !g.off || g.y_f32 || g.cols < 2048 || g.ldw % 2048 ? 0 : (grp * 13 + row0 / kGwM) % (g.cols / kGtBK);
}

template <int BM, int BN, int WGM, int WGN>
__global__ __launch_bounds__(64 * WGM * WGN, (WGM * WGN > 4 ? 1 : BM + BN <= 192 ? 3 : 2)) void group_tile_kernel(pi_group_gemm g, int nx, int max_units) {
    using Tile = GemmTile<bf16, BM, BN, WGM, WGN>;
    constexpr int WM = Tile::WM, WN = Tile::WN, MT = Tile::MT, NT = Tile::NT;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tt = (g.T + BN - 1) / BN;                       // token tiles of a group without a list
    const int units = g.off ? *g.n_tiles * nx : max_units;
    const int per = (units + 7) / 8, unit = (int)(blockIdx.x % 8) * per + (int)blockIdx.x / 8;
    if ((int)blockIdx.x / 8 >= per || unit >= units) return;
    const int tx = unit % nx, ty = unit / nx;
    int grp, lo, n;                                           // group, first token (place), tokens from there on
    if (g.off) {
        const int2 t = reinterpret_cast<const int2 *>(g.tiles)[ty];
        grp = t.x; lo = t.y; n = g.off[grp + 1] - lo;
    } else {
        grp = ty / tt; lo = (ty % tt) * BN; n = g.T - lo;
    }
    n = min(n, BN);
    const int row0 = tx * BM;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const int wm = wave % WGM, wn = wave / WGM;
    const bf16 * W = (const bf16 *)g.W + (size_t)grp * g.w_gs;
    const bf16 * x = (const bf16 *)g.x + (g.off ? 0 : (size_t)grp * g.x_gs);
    const bf16 * ga[Tile::ACH]; const bf16 * gb[Tile::BCH];
#pragma unroll
    for (int j = 0; j < Tile::ACH; ++j) ga[j] = W + (size_t)min(row0 + Tile::chunk_row(j), g.rows - 1) * g.ldw + Tile::chunk_col();
#pragma unroll
    for (int j = 0; j < Tile::BCH; ++j) {
        const int s = lo + min(Tile::chunk_row(j), n - 1);
        gb[j] = x + (size_t)(g.gather ? g.gather[s] / g.gather_div : s) * g.ldx + Tile::chunk_col();
    }
    pi_f4 acc[MT][NT];
    Tile::run(smem, ga, gb, g.cols / kGtBK, acc, group_first(g, grp, row0));
    group_store(g, grp, lo, n, row0 + wm * WM, wn * WN, q, i, acc);
}

// The same through LDS (store_turned), one kind of epilogue at a time: the code runs once a unit and its instructions come from L2 each time.
enum { kStorePlain, kStoreRelu2, kStoreGlu };
template <int KIND, int MT, int NT>
__device__ __forceinline__ void group_store_turned(const pi_group_gemm & g, int grp, int lo, int n, int row0, int tok0, int lane, const pi_f4 (&acc)[MT][NT], unsigned char * turn) {
    asm volatile("" : "+v"(lane));                     // what follows is computed here, not kept in registers across the products
    const float one = g.glu_plain_up ? 0.0f : 1.0f;
    const int out0 = KIND == kStoreGlu ? row0 / 2 : row0, outs = KIND == kStoreGlu ? g.rows / 2 : g.rows;
#pragma unroll
    for (int nn = 0; nn < NT; ++nn) {
        const float alpha = g.pair_w ? g.alpha * g.pair_w[g.gather[lo + min(tok0 + nn * 16 + (lane & 15), n - 1)]] : g.alpha;
        __builtin_amdgcn_sched_barrier(0);
        uint2 out[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if constexpr (KIND == kStoreGlu) {
                const bf16 v[2] = {(bf16)clamped_glu(acc[m][nn][0] * alpha, acc[m][nn][1] * alpha, g.glu_limit, g.glu_gain, one),
                                   (bf16)clamped_glu(acc[m][nn][2] * alpha, acc[m][nn][3] * alpha, g.glu_limit, g.glu_gain, one)};
                out[m].x = __builtin_bit_cast(uint32_t, v);
            } else {
                bf16 b[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = acc[m][nn][r] * alpha;
                    if (KIND == kStoreRelu2) { v = fmaxf(v, 0.0f); v *= v; }
                    b[r] = (bf16)v;
                }
                out[m] = __builtin_bit_cast(uint2, b);
            }
        }
        store_turned<KIND == kStoreGlu ? 4 : 8>(out, turn, lane, [&](int t, int piece) -> void * {
            const int to = tok0 + nn * 16 + t;
            return to < n && out0 + piece * 8 < outs ? (bf16 *)g.y + (g.off ? 0 : (size_t)grp * g.y_gs) + (size_t)(lo + to) * g.ldy + out0 + piece * 8 : nullptr;
        });
    }
}

constexpr long long kGwValues = 1LL << 31;                          // of a group's matrix: off_a counts its bytes in 32 bits
// the same product in the large tiles of gemm_wide.  256 rows by 128 tokens, or 128 by 256: an expert of more than 128 tokens then has its weights
// read once, and by one workgroup.  64 experts, both products, us, tiles of 128 / 256 tokens: 192 tokens an expert on average 407 -> 390 (1408 x 4096), 624 -> 585
// (with a gate); 8 experts of 140, 4096 x 4096 with a gate 245 -> 176; of 96 tokens 290 and 334.
template <int M, int N, bool LIST> struct GroupProduct {
    static constexpr bool kPairs = false, kList = false, kTurned = false;
    static constexpr int kM = M, kN = N;
    const pi_group_gemm & g;
    int nk, tt;                                                     // tt: token tiles of a group without a list
    bool whole;
    __device__ __forceinline__ WidePlace place(const WideDeal & deal, int c) const {
        WidePlace p;
        int ty;
        deal.unit(c, ty, p.row0, p.rows);
        if (LIST) {
            const int2 t = reinterpret_cast<const int2 *>(g.tiles)[ty];
            p.grp = t.x; p.lo = t.y; p.n = g.off[p.grp + 1] - p.lo;
        } else {
            p.grp = ty / tt; p.lo = (ty % tt) * N; p.n = g.T - p.lo;
        }
        p.n = min(p.n, N);
        return p;
    }
    __device__ __forceinline__ bool read_once(const WidePlace & p) const { return LIST && g.off[p.grp + 1] - g.off[p.grp] <= N; }
    __device__ __forceinline__ int first(const WidePlace & p) const { return LIST ? group_first(g, p.grp, p.row0) : 0; }
    __device__ __forceinline__ const unsigned char * base_a(const WidePlace & p, int) const { return (const unsigned char *)((const bf16 *)g.W + (size_t)p.grp * g.w_gs); }
    __device__ __forceinline__ const unsigned char * base_b(const WidePlace & p) const { return (const unsigned char *)((const bf16 *)g.x + (g.off ? 0 : (size_t)p.grp * g.x_gs)); }
    __device__ __forceinline__ uint32_t off_a(const WidePlace & p, int r) const { return (uint32_t)(p.row0 + r) * (uint32_t)(g.ldw * 2); }
    __device__ __forceinline__ size_t off_b(const WidePlace & p, int r) const { return (size_t)(g.gather ? g.gather[p.lo + r] / g.gather_div : p.lo + r) * (size_t)g.ldx * 2; }
    template <int MT> __device__ __forceinline__ void store(const WidePlace & p, int rb, int tb, const pi_f4 (&acc)[MT][4], unsigned char * turn, int lane) const {
        if (whole && g.glu) group_store_turned<kStoreGlu>(g, p.grp, p.lo, p.n, p.row0 + rb, tb, lane, acc, turn);
        else if (whole && g.relu2) group_store_turned<kStoreRelu2>(g, p.grp, p.lo, p.n, p.row0 + rb, tb, lane, acc, turn);
        else if (whole) group_store_turned<kStorePlain>(g, p.grp, p.lo, p.n, p.row0 + rb, tb, lane, acc, turn);
        else group_store(g, p.grp, p.lo, p.n, p.row0 + rb, tb, lane >> 4, lane & 15, acc);
    }
};
// n_tiles: token tiles of a product without a list.  LIST: g.off; the two are kernels of their own because a choice of the hint at run time costs the copying
// waves what matters to units that share their weights (22016 x 4096 by 400 tokens: 83 -> 88 us).
template <int M, int N, bool LIST>
__global__ __launch_bounds__(512, 1) void group_wide_kernel(pi_group_gemm g, int n_tiles) {
    extern __shared__ __align__(16) unsigned char smem[];
    const GroupProduct<M, N, LIST> prod{g, g.cols / kGtBK, (g.T + N - 1) / N, !g.y_f32 && g.rows % (g.glu ? 16 : 8) == 0 && g.ldy % 8 == 0 && g.y_gs % 8 == 0};
    gemm_wide<bf16>(prod, WideDeal(g.rows, LIST ? *g.n_tiles : n_tiles, g.n_group > 1 ? 1 : kGwBand, M), smem);       // (bands of experts' tiles measured no better)
}

template <int M, int N, bool LIST> int launch_group_wide(const pi_group_gemm & g, hipStream_t st) {
    static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&group_wide_kernel<M, N, LIST>), hipFuncAttributeMaxDynamicSharedMemorySize, kGwLds);
    if (raised != hipSuccess) return pi::hip_fail(raised, "group_wide: LDS size");
    const long long tiles = LIST ? g.max_tiles : (long long)g.n_group * ((g.T + N - 1) / N), units = tiles * ((g.rows + M - 1) / M);
    if (units > (1 << 30)) return pi::fail(PI_E_ARG, "pi_k_group_gemm_tile: too many tiles");
    hipLaunchKernelGGL((group_wide_kernel<M, N, LIST>), dim3(wide_blocks(units)), dim3(512), kGwLds, st, g, (int)tiles);
    return pi::check_launch("pi_k_group_gemm_tile");
}

template <int BM, int BN, int WGM, int WGN> int launch_group_tile(const pi_group_gemm & g, hipStream_t st) {
    using Tile = GemmTile<bf16, BM, BN, WGM, WGN>;
    static bool raised = false;
    if (!raised && Tile::kLds > 64 * 1024) {
        PI_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&group_tile_kernel<BM, BN, WGM, WGN>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)Tile::kLds));
        raised = true;
    }
    const int nx = (g.rows + BM - 1) / BM;
    const long long units = (long long)nx * (g.off ? g.max_tiles : (long long)g.n_group * ((g.T + BN - 1) / BN));
    if (units > (1 << 30)) return pi::fail(PI_E_ARG, "pi_k_group_gemm_tile: too many tiles");
    hipLaunchKernelGGL((group_tile_kernel<BM, BN, WGM, WGN>), dim3((unsigned)((units + 7) / 8 * 8)), dim3(64 * WGM * WGN), Tile::kLds, st, g, nx, (int)units);
    return pi::check_launch("pi_k_group_gemm_tile");
}

template <typename ST>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float * __restrict__ x, const float * __restrict__ mix, const ST * __restrict__ y,
                                                          const int32_t * __restrict__ inv, const float * __restrict__ weights, int top, int cols,
                                                          float * __restrict__ out, float * __restrict__ keep) {
    const int t = blockIdx.y, c0 = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (c0 >= cols) return;
    if ((cols & 3) == 0) {                           // four columns a thread
        const size_t o = (size_t)t * cols + c0;
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (weights) for (int k = 0; k < top; ++k) {
            const float w = weights[(size_t)t * top + k];
            struct alignas(4 * sizeof(ST)) Quad { ST v[4]; };
            const Quad q = *reinterpret_cast<const Quad *>(y + (size_t)inv[(size_t)t * top + k] * cols + c0);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = fmaf(w, from_st(q.v[j]), s[j]);
        }
        const float4 a = *reinterpret_cast<const float4 *>(x + o), b = *reinterpret_cast<const float4 *>(mix + o);
        const float4 v = make_float4(a.x + (b.x + s[0]), a.y + (b.y + s[1]), a.z + (b.z + s[2]), a.w + (b.w + s[3]));
        *reinterpret_cast<float4 *>(out + o) = v;
        if (keep) *reinterpret_cast<float4 *>(keep + o) = v;
        return;
    }
    for (int c = c0; c < min(c0 + 4, cols); ++c) {
        const size_t o = (size_t)t * cols + c;
        float s = 0.0f;
        if (weights) for (int k = 0; k < top; ++k) s = fmaf(weights[(size_t)t * top + k], from_st(y[(size_t)inv[(size_t)t * top + k] * cols + c]), s);
        const float v = x[o] + (mix[o] + s);
        out[o] = v;
        if (keep) keep[o] = v;
    }
}

__global__ void pad_cols_kernel(const uint16_t * __restrict__ in, int64_t rows, int cols, uint16_t * __restrict__ out, int ld) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < rows * ld; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / ld; const int c = (int)(i % ld);
        out[i] = c < cols ? in[r * cols + c] : (uint16_t)0;
    }
}
__global__ void place_kernel(const uint16_t * __restrict__ in, int64_t rows, int cols, uint16_t * __restrict__ out, int ld, int col0, int width, int64_t row0, int row_step) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < rows * width; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / width; const int c = (int)(i % width);
        out[(size_t)(row0 + r * row_step) * ld + col0 + c] = c < cols ? in[r * cols + c] : (uint16_t)0;
    }
}
__global__ void transpose_pad_kernel(const uint16_t * __restrict__ in, int n_mat, int rows, int cols, uint16_t * __restrict__ out, int ld) {
    const int64_t n = (int64_t)n_mat * cols * ld;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(i % ld); const int64_t mc = i / ld;
        const int64_t mat = mc / cols; const int c = (int)(mc % cols);
        out[i] = r < rows ? in[(mat * rows + r) * cols + c] : (uint16_t)0;
    }
}

__global__ void cells_advance_kernel(int T, const int32_t * __restrict__ seq, const int32_t * __restrict__ lists, size_t list_ld, int32_t * __restrict__ n_vis,
                                     int32_t * __restrict__ cell, int32_t * step) {
    const int t = threadIdx.x;
    if (t < T) {
        const int n = n_vis[t] + 1;
        n_vis[t] = n;
        cell[t] = lists[(size_t)seq[t] * list_ld + min((size_t)n, list_ld) - 1];        // (behind the last step of a full pool: not used)
    }
    if (t == 0) *step += 1;
}

}  // namespace

namespace pi {
int pass_start(const PassStart & p, hipStream_t st) {
    const int nt = p.norm ? embed_norm_block(p.cols) : 256;
    const auto blocks = [&](size_t n) { return (int)((n + nt - 1) / nt); };
    const int embeds = p.table ? p.T : 0, copies = blocks((p.words + 3) / 4), appends = blocks((size_t)p.n_append);
    int rots = 0;
    for (int k = 0; k < p.n_rot; ++k) rots += blocks((size_t)p.T * (p.rot[k].dims / 2));
    if (embeds + copies + appends + rots == 0) return PI_OK;
    const Bigram g{(const uint16_t *)p.table, p.scale, (const uint16_t *)p.bigram, p.buckets, (long long)p.mul_prev, (long long)p.mul_cur};
    hipLaunchKernelGGL(pass_start_kernel, dim3(embeds + copies + appends + rots), dim3(nt), 0, st, p, g, embeds, copies, appends);
    return check_launch("pass_start");
}
}  // namespace pi

extern "C" {

int pi_k_embed_norm(const void * table, int cols, const int32_t * tokens, int T, const float * w, float eps, float * x, pi_stream_t stream) {
    if (!table || !tokens || !w || !x || cols <= 0 || T <= 0) return pi::fail(PI_E_ARG, "pi_k_embed_norm: bad arguments");
    hipLaunchKernelGGL(embed_norm_kernel, dim3(T), dim3(embed_norm_block(cols)), 0, (hipStream_t)stream, (const uint16_t *)table, cols, tokens, w, eps, x);
    return pi::check_launch("pi_k_embed_norm");
}

int pi_k_embed_bigram(const void * table, int cols, const int32_t * tokens, int32_t * prev, int T, float scale, const void * bigram, int32_t buckets, int64_t mul_prev,
                      int64_t mul_cur, int carry, float * x, float * x0, pi_stream_t stream) {
    if (!table || !tokens || !prev || !x || cols <= 0 || T <= 0 || (bigram && buckets <= 0)) return pi::fail(PI_E_ARG, "pi_k_embed_bigram: bad arguments");
    hipLaunchKernelGGL(embed_bigram_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, Bigram{(const uint16_t *)table, scale, (const uint16_t *)bigram, buckets, (long long)mul_prev, (long long)mul_cur},
                       cols, tokens, prev, carry, x, x0);
    return pi::check_launch("pi_k_embed_bigram");
}

int pi_k_layer_norm(int type, float * x, const int32_t * rows, int T, int cols, float eps, const float * w, const float * x0, const float * step, void * out, int ld, int ol,
                    pi_stream_t stream) {
    if (!x || !w || !out || T <= 0 || cols <= 0 || ld < cols || (rows && (x0 || step))) return pi::fail(PI_E_ARG, "pi_k_layer_norm: bad arguments");
    if (ol && (type != PI_TYPE_BF16 || T > kBtMaxT || ld % 8)) return pi::fail(PI_E_ARG, "pi_k_layer_norm: operand layout needs BF16, T <= 16, ld % 8 == 0");
    const int block = cols > 2048 ? 1024 : cols > 512 ? 512 : 256;
    if (type == PI_TYPE_BF16) hipLaunchKernelGGL(layer_norm_kernel<bf16>, dim3(T), dim3(block), 0, (hipStream_t)stream, x, rows, cols, eps, w, x0, step, (bf16 *)out, ld, ol);
    else if (type == PI_TYPE_F32) hipLaunchKernelGGL(layer_norm_kernel<float>, dim3(T), dim3(block), 0, (hipStream_t)stream, x, rows, cols, eps, w, x0, step, (float *)out, ld, 0);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_layer_norm: type");
    return pi::check_launch("pi_k_layer_norm");
}

int pi_k_res_norm(int type, const pi_res_norm * p, pi_stream_t stream) {
    if (!p || !p->x || !p->out || p->T <= 0 || p->cols <= 0 || (p->mix && p->gate_z && (!p->gate_b || p->off_gate < 0 || p->off_gate + p->cols > p->ld_gate)) || (p->h && p->ld < p->cols))
        return pi::fail(PI_E_ARG, "pi_k_res_norm: bad arguments");
    if (p->h && p->ol && (type != PI_TYPE_BF16 || p->T > kBtMaxT || p->ld % 8)) return pi::fail(PI_E_ARG, "pi_k_res_norm: operand layout needs BF16, T <= 16, ld % 8 == 0");
    if (type == PI_TYPE_BF16) return launch_res_norm<bf16>(*p, (hipStream_t)stream);
    if (type == PI_TYPE_F32) return launch_res_norm<float>(*p, (hipStream_t)stream);
    return pi::fail(PI_E_UNSUPPORTED, "pi_k_res_norm: type");
}

int pi_k_ffn_front(int type, const float * z, int ldz, int T, const pi_ffn_front * front, pi_stream_t stream) {
    if (!z || !front || T <= 0 || !front_ok(*front, ldz)) return pi::fail(PI_E_ARG, "pi_k_ffn_front: bad arguments");
    const int per = front_blocks(*front);
    if (per == 0) return PI_OK;
    if ((long long)per * T > (1 << 30)) return pi::fail(PI_E_ARG, "pi_k_ffn_front: too many tokens");
    if (type == PI_TYPE_BF16) hipLaunchKernelGGL(ffn_front_kernel<bf16>, dim3(per * T), dim3(256), front_lds_bytes(*front), (hipStream_t)stream, *front, z, ldz, per);
    else if (type == PI_TYPE_F32) hipLaunchKernelGGL(ffn_front_kernel<float>, dim3(per * T), dim3(256), front_lds_bytes(*front), (hipStream_t)stream, *front, z, ldz, per);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_ffn_front: type");
    return pi::check_launch("pi_k_ffn_front");
}

int pi_k_norm_pair(int type, const float * x, const int32_t * rows, int T, int cols, float eps, const float * wa, void * out_a,
                   const float * wb, void * out_b, int ld, int ol, pi_stream_t stream) {
    if (!x || !wa || !out_a || (wb && !out_b) || T <= 0 || cols <= 0 || ld < cols) return pi::fail(PI_E_ARG, "pi_k_norm_pair: bad arguments");
    if (ol && (type != PI_TYPE_BF16 || T > kBtMaxT || ld % 8)) return pi::fail(PI_E_ARG, "pi_k_norm_pair: operand layout needs BF16, T <= 16, ld % 8 == 0");
    if (T > kBtMaxT && cols % 4 == 0 && cols > 512 && cols <= 4096 && ld % 4 == 0 && (((uintptr_t)x | (uintptr_t)wa | (uintptr_t)wb | (uintptr_t)out_a | (uintptr_t)out_b) & 15) == 0 && (type == PI_TYPE_BF16 || type == PI_TYPE_F32)) {
        if (type == PI_TYPE_BF16) hipLaunchKernelGGL(norm_pair_quads_kernel<bf16>, dim3(T), dim3(256), 0, (hipStream_t)stream, x, rows, cols, eps, wa, (bf16 *)out_a, wb, (bf16 *)out_b, ld);
        else hipLaunchKernelGGL(norm_pair_quads_kernel<float>, dim3(T), dim3(256), 0, (hipStream_t)stream, x, rows, cols, eps, wa, (float *)out_a, wb, (float *)out_b, ld);
        return pi::check_launch("pi_k_norm_pair");
    }
    const int block = cols > 2048 ? 1024 : cols > 512 ? 512 : 256;
    if (type == PI_TYPE_BF16)
        hipLaunchKernelGGL(norm_pair_kernel<bf16>, dim3(T), dim3(block), 0, (hipStream_t)stream, x, rows, cols, eps, wa, (bf16 *)out_a, wb, (bf16 *)out_b, ld, ol);
    else if (type == PI_TYPE_F32)
        hipLaunchKernelGGL(norm_pair_kernel<float>, dim3(T), dim3(block), 0, (hipStream_t)stream, x, rows, cols, eps, wa, (float *)out_a, wb, (float *)out_b, ld, 0);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_norm_pair: type");
    return pi::check_launch("pi_k_norm_pair");
}

int pi_k_group_gemm(int type, const pi_group_gemm * g, pi_stream_t stream) {
    if (!g || !g->W || !g->x || !g->y || g->rows <= 0 || g->cols <= 0 || g->cols % 32 || g->ldw < g->cols || g->ldw % 8 || g->ldx < g->cols || g->ldx % 8 ||
        g->ldy < (g->glu ? g->rows / 2 : g->rows) || (g->glu && (g->rows % 2 || g->relu2)) || g->T <= 0 || g->n_group <= 0 || g->n_group > 65535 || (g->gather && g->gather_div <= 0) || (g->pair_w && (!g->gather || !g->off)) || g->w_gs % 8 || g->x_gs % 8)
        return pi::fail(PI_E_ARG, "pi_k_group_gemm: bad arguments");
    const dim3 grid((g->rows + 63) / 64, (g->T + 31) / 32, g->n_group);
    if (grid.y > 65535) return pi::fail(PI_E_ARG, "pi_k_group_gemm: too many tokens");
    if (type == PI_TYPE_BF16) hipLaunchKernelGGL(group_gemm_kernel<bf16>, grid, dim3(256), 0, (hipStream_t)stream, *g);
    else if (type == PI_TYPE_F32) hipLaunchKernelGGL(group_gemm_kernel<float>, grid, dim3(256), 0, (hipStream_t)stream, *g);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_group_gemm: type");
    return pi::check_launch("pi_k_group_gemm");
}

int pi_k_rope_angles(const int32_t * pos, int T, int dims, double base, void * cs, pi_stream_t stream) {
    if (!pos || !cs || T <= 0 || dims <= 0 || dims % 2 || !(base > 0.0)) return pi::fail(PI_E_ARG, "pi_k_rope_angles: bad arguments");
    hipLaunchKernelGGL(rope_angles_kernel, dim3((T * (dims / 2) + 63) / 64), dim3(64), 0, (hipStream_t)stream, pos, T, dims, base, (float2 *)cs);
    return pi::check_launch("pi_k_rope_angles");
}

int pi_k_rope_angles_table(const int32_t * pos, int T, int dims, const double * freq, double length, void * cs, pi_stream_t stream) {
    if (!pos || !cs || !freq || T <= 0 || dims <= 0 || dims % 2) return pi::fail(PI_E_ARG, "pi_k_rope_angles_table: bad arguments");
    hipLaunchKernelGGL(rope_table_kernel, dim3((T * (dims / 2) + 63) / 64), dim3(64), 0, (hipStream_t)stream, pos, T, dims / 2, freq, length, (float2 *)cs);
    return pi::check_launch("pi_k_rope_angles_table");
}

int pi_k_router_parts(int T, int n_expert, int cols) {
    return T > kBtMaxT && n_expert > 0 && n_expert <= kRouterExperts && cols > 0 && cols % kRouterCols == 0 && cols / kRouterCols <= 65535 ? cols / kRouterCols : 0;
}

int pi_k_route_long(const void * router, int n_expert, int cols, const void * x, int T, float * parts, int n_top, int n_group, int n_keep, const float * bias, int32_t * ids, float * weights,
                    pi_stream_t stream) {
    const int n = pi_k_router_parts(T, n_expert, cols);
    if (!n) return pi::fail(PI_E_UNSUPPORTED, "pi_k_route_long: more than 16 tokens, up to 128 experts, columns in 512s");
    if (!router || !x || !parts || !ids || !weights || (((uintptr_t)router | (uintptr_t)x) & 15) || n_top <= 0 || n_group <= 0 || n_expert % n_group || n_keep <= 0 || n_keep > n_group ||
        n_top > n_keep * (n_expert / n_group) || (!bias && n_group != 1))
        return pi::fail(PI_E_ARG, "pi_k_route_long: bad arguments");
    const size_t lds = (size_t)(n_expert + 15) / 16 * 16 * kRouterPitch;
    static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&router_parts_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kRouterExperts * kRouterPitch);
    if (raised != hipSuccess) return pi::hip_fail(raised, "pi_k_route_long: LDS size");
    hipLaunchKernelGGL(router_parts_kernel, dim3((T + 63) / 64, n), dim3(256), lds, (hipStream_t)stream, (const bf16 *)router, n_expert, cols, (const bf16 *)x, T, parts);
    RouteArgs r{parts, n_expert, n_top, n_group, n_keep, bias, ids, weights};
    r.raw = !bias; r.parts = n; r.part_ld = (size_t)T * n_expert;
    hipLaunchKernelGGL(route_kernel, dim3(T), dim3(n_expert > 64 ? 128 : 64), route_lds_bytes(n_expert, n_group, n_top), (hipStream_t)stream, r);
    return pi::check_launch("pi_k_route_long");
}

int pi_k_route_scores(const float * z, int T, int n_expert, int n_top, int32_t * ids, float * weights, pi_stream_t stream) {
    if (!z || !ids || !weights || T <= 0 || n_expert <= 0 || n_expert > 4096 || n_top <= 0 || n_top > n_expert) return pi::fail(PI_E_ARG, "pi_k_route_scores: bad arguments");
    RouteArgs r{z, n_expert, n_top, 1, 1, nullptr, ids, weights};
    r.raw = true;
    hipLaunchKernelGGL(route_kernel, dim3(T), dim3(n_expert > 128 ? 256 : n_expert > 64 ? 128 : 64), route_lds_bytes(n_expert, 1, n_top), (hipStream_t)stream, r);
    return pi::check_launch("pi_k_route_scores");
}

int pi_k_route(const float * z, int T, int n_expert, int n_top, int n_group, int n_keep, const float * bias, int32_t * ids, float * weights, pi_stream_t stream) {
    if (!z || !bias || !ids || !weights || T <= 0 || n_expert <= 0 || n_expert > 4096 || n_top <= 0 || n_group <= 0 || n_expert % n_group || n_keep <= 0 || n_keep > n_group ||
        n_top > n_keep * (n_expert / n_group))
        return pi::fail(PI_E_ARG, "pi_k_route: bad arguments");
    hipLaunchKernelGGL(route_kernel, dim3(T), dim3(n_expert > 128 ? 256 : n_expert > 64 ? 128 : 64), route_lds_bytes(n_expert, n_group, n_top), (hipStream_t)stream, RouteArgs{z, n_expert, n_top, n_group, n_keep, bias, ids, weights});
    return pi::check_launch("pi_k_route");
}

int pi_k_moe_sort(const int32_t * ids, int n_pairs, int n_expert, int32_t * off, int32_t * perm, int32_t * inv, int tile_n, int32_t * tiles, int32_t * n_tiles,
                  pi_stream_t stream) {
    if (!ids || !off || !perm || !inv || n_pairs <= 0 || n_expert <= 0 || n_expert > 8192 || (tiles && (tile_n <= 0 || !n_tiles))) return pi::fail(PI_E_ARG, "pi_k_moe_sort: bad arguments");
    hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), sizeof(int) * n_expert, (hipStream_t)stream, ids, n_pairs, n_expert, off, perm, inv, tile_n, (int2 *)tiles, n_tiles);
    return pi::check_launch("pi_k_moe_sort");
}

// what both forms below ask of their operands
static int group_tile_args(const pi_group_gemm * g) {
    if (!g || !g->W || !g->x || !g->y || g->rows <= 0 || g->cols <= 0 || g->cols % kGtBK || g->ldw < g->cols || g->ldw % 8 || g->ldx < g->cols || g->ldx % 8 ||
        g->ldy < (g->glu ? g->rows / 2 : g->rows) || (g->glu && (g->rows % 2 || g->relu2)) || g->T <= 0 || g->n_group <= 0 || (g->gather && g->gather_div <= 0) || (g->pair_w && (!g->gather || !g->off)) || g->w_gs % 8 || g->x_gs % 8 || (g->off && (!g->tiles || !g->n_tiles || g->max_tiles <= 0)))
        return pi::fail(PI_E_ARG, "pi_k_group_gemm_tile: bad arguments");
    if ((((uintptr_t)g->W | (uintptr_t)g->x | (uintptr_t)g->y) & 15) != 0) return pi::fail(PI_E_ARG, "pi_k_group_gemm_tile: operands must be 16-byte aligned");
    return PI_OK;
}

int pi_k_group_gemm_tile(const pi_group_gemm * g, int tile_n, pi_stream_t stream) {
    const int rc = group_tile_args(g);
    if (rc != PI_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    // 256-row tiles from the second half on, and at least four stages for a unit's ends to hide behind: measured as fast or faster at every number of
    // tokens and groups from there on (32 heads' 256 x 512 products of 128 tokens: 11.4 us both; 4096 x 512 by 2048 tokens 20.6 -> 16.1)
    if (tile_n == 128 && g->rows > 128 && g->cols >= 4 * kGtBK && (long long)g->rows * g->ldw < kGwValues)
        return g->off ? launch_group_wide<kGwM, kGwN, true>(*g, st) : launch_group_wide<kGwM, kGwN, false>(*g, st);
    if (tile_n == 128) return launch_group_tile<128, 128, 2, 2>(*g, st);
    if (tile_n == 64) return g->rows <= 64 ? launch_group_tile<64, 64, 2, 2>(*g, st) : launch_group_tile<128, 64, 2, 2>(*g, st);
    return pi::fail(PI_E_ARG, "pi_k_group_gemm_tile: tile_n must be 64 or 128");
}

// Tokens per tile, by the tokens an expert has on average (multinomial counts).  Experts' matrices of 512 MB and more (2 MB a compute unit) go through
// the large tiles whatever the number: a workgroup streams them at the memory's rate, and 64 and 128 x 128 tiles do not.  Both products of five shapes
// (experts x ff x width, * with a gate; us in tiles of 64, 128 and 256 tokens at 16 / 64 / 160 tokens): 64 x 1408 x 4096 272, 249, 283 / 359, 279,
// 324 / 573, 404, 378; the same * 390, 342, 420 / 517, 393, 473 / 879, 607, 560; 64 x 1408 x 2048 * 205, 179, 229 / 264, 211, 257 / 419, 319, 306;
// 8 x 4096 x 4096 * 151, 134, 147 / 211, 138, 152 / 433, 248, 180; 160 x 1536 x 5120 900, 817, 983 at 16.  Less than that, 16 x 1408 x 2048 *, 32 x 1024 x 1024
// and 64 x 256 x 1024 *: at 16 tokens 55, 57, 31, 35 and 27, 29 in tiles of 64 and 128, so 64 until they start to need two an expert, which is at
// 52 tokens; in tiles of 128 and 256 at 150 tokens 94, 87, 43, 45 and 48, 47, at 192 82, 93, 45, 49 and 46, 50.
int pi_k_expert_tile(int64_t n_pairs, int n_expert, int up_rows, int up_ld, int down_rows, int down_ld) {
    const int64_t up = (int64_t)up_rows * up_ld, down = (int64_t)down_rows * down_ld;
    const bool large = 2 * n_expert * (up + down) >= 512LL << 20 && up_rows > 128 && down_rows > 128 && up_ld >= 4 * kGtBK && down_ld >= 4 * kGtBK;
    // (beyond kGwValues an expert's matrix has no tiles of 256 tokens, and those of 128 go another way)
    return large && n_pairs > 132LL * n_expert && up < kGwValues && down < kGwValues ? 256 : large || n_pairs > 52LL * n_expert ? 128 : 64;
}

int pi_k_group_gemm_tall(const pi_group_gemm * g, pi_stream_t stream) {
    const int rc = group_tile_args(g);
    if (rc != PI_OK) return rc;
    if (!g->off || g->rows <= 64 || g->cols < 4 * kGtBK || (long long)g->rows * g->ldw >= kGwValues)
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_group_gemm_tall: lists of more than 64 rows, at least 256 columns and less than 2^31 values a group");
    return launch_group_wide<128, 256, true>(*g, (hipStream_t)stream);
}

int pi_k_moe_combine(int type, const float * x, const float * mix, const void * y, const int32_t * inv, const float * weights, int n_top, int T, int cols,
                     float * out, float * keep, pi_stream_t stream) {
    if (!x || !mix || !out || T <= 0 || T > 65535 || cols <= 0 || (weights && (!y || !inv || n_top <= 0))) return pi::fail(PI_E_ARG, "pi_k_moe_combine: bad arguments");
    const dim3 grid((cols + 1023) / 1024, T);
    if (type == PI_TYPE_BF16) hipLaunchKernelGGL(moe_combine_kernel<bf16>, grid, dim3(256), 0, (hipStream_t)stream, x, mix, (const bf16 *)y, inv, weights, n_top, cols, out, keep);
    else hipLaunchKernelGGL(moe_combine_kernel<float>, grid, dim3(256), 0, (hipStream_t)stream, x, mix, (const float *)y, inv, weights, n_top, cols, out, keep);
    return pi::check_launch("pi_k_moe_combine");
}

int pi_k_pad_cols_bf16(const void * in, int64_t rows, int cols, void * out, int ld, pi_stream_t stream) {
    if (!in || !out || rows <= 0 || cols <= 0 || ld < cols) return pi::fail(PI_E_ARG, "pi_k_pad_cols_bf16: bad arguments");
    hipLaunchKernelGGL(pad_cols_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, (const uint16_t *)in, rows, cols, (uint16_t *)out, ld);
    return pi::check_launch("pi_k_pad_cols_bf16");
}

int pi_k_place_bf16(const void * in, int64_t rows, int cols, void * out, int ld, int col0, int width, int64_t row0, int row_step, pi_stream_t stream) {
    if (!in || !out || rows <= 0 || cols <= 0 || width < cols || col0 < 0 || col0 + width > ld || row0 < 0 || row_step <= 0) return pi::fail(PI_E_ARG, "pi_k_place_bf16: bad arguments");
    hipLaunchKernelGGL(place_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, (const uint16_t *)in, rows, cols, (uint16_t *)out, ld, col0, width, row0, row_step);
    return pi::check_launch("pi_k_place_bf16");
}

int pi_k_transpose_pad_bf16(const void * in, int n_mat, int rows, int cols, void * out, int ld, pi_stream_t stream) {
    if (!in || !out || n_mat <= 0 || rows <= 0 || cols <= 0 || ld < rows) return pi::fail(PI_E_ARG, "pi_k_transpose_pad_bf16: bad arguments");
    hipLaunchKernelGGL(transpose_pad_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, (const uint16_t *)in, n_mat, rows, cols, (uint16_t *)out, ld);
    return pi::check_launch("pi_k_transpose_pad_bf16");
}

int pi_k_cells_advance(int T, const int32_t * seq, const int32_t * lists, size_t list_ld, int32_t * n_vis, int32_t * cell, int32_t * step, pi_stream_t stream) {
    if (T <= 0 || T > 64 || !seq || !lists || !n_vis || !cell || !step) return pi::fail(PI_E_ARG, "pi_k_cells_advance: bad arguments");
    hipLaunchKernelGGL(cells_advance_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, T, seq, lists, list_ld, n_vis, cell, step);
    return pi::check_launch("pi_k_cells_advance");
}

}  // extern "C"
