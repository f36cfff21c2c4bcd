// Steps of up to 16 tokens of a model described layer by layer (bf16), as few launches as its dependencies allow: everything behind
// the joint projection (absorbed queries, rotation, cells, expert choice) in one, the merge of a split attention with the value
// expansion together with the experts' first matrices in one, and one for what closes a layer - attention output and the experts' second
// matrices as a single long dot product per row, plus the residual.
#include "layer_types.hpp"
#include "mixers.hpp"
#include "route.hpp"

namespace {

constexpr int kRopePerWg = 512;           // rotated query pairs of a workgroup
// Behind the joint projection: per head the absorbed query (64 latent rows a workgroup), per token the rotated query parts, the cell,
// and the expert choice.
__global__ __launch_bounds__(256) void latent_step_kernel(pi_latent_prep p, const uint16_t * __restrict__ uk_t, RouteArgs r, int n_absorb) {
    extern __shared__ __align__(16) float sm[];
    __shared__ double red[4];
    const int hd = p.dim + p.rot_dim, half = p.rot_dim / 2, tid = threadIdx.x;
    int b = blockIdx.x;
    if (b < n_absorb) {                                       // a head's query in latent coordinates: 64 rows of W_uk^T against the step's tokens
        const int tiles = (p.kv_rank + 63) / 64, h = b / tiles, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
        const int row0 = (b % tiles) * 64 + wave * 16;
        if (row0 >= p.kv_rank) return;
        const uint16_t * W = uk_t + ((size_t)h * p.kv_rank + min(row0 + i, p.kv_rank - 1)) * p.dim_ld + g * 8;
        const float * z = p.z + (size_t)min(i, p.T - 1) * p.ldz + h * hd;
        const bool whole = p.dim % 8 == 0 && hd % 4 == 0 && p.ldz % 4 == 0;        // eight columns are two 16-byte loads
        pi_f4 acc = pi_f4{0, 0, 0, 0};
        for (int k0 = 0; k0 < p.dim_ld; k0 += 128) {          // four steps requested together, unguarded; what is past the end is zeroed
            pi_u32x4 w[4];
            float q[4][8];
#pragma unroll
            for (int s = 0; s < 4; ++s) w[s] = pi_ld16(W + min(k0 + s * 32, p.dim_ld - 32));
            if (whole) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const float4 * zp = reinterpret_cast<const float4 *>(z + min(k0 + s * 32 + g * 8, p.dim - 8));
                    const float4 a = zp[0], c = zp[1];
                    q[s][0] = a.x; q[s][1] = a.y; q[s][2] = a.z; q[s][3] = a.w; q[s][4] = c.x; q[s][5] = c.y; q[s][6] = c.z; q[s][7] = c.w;
                }
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int j = 0; j < 8; ++j) q[s][j] = z[min(k0 + s * 32 + g * 8 + j, p.dim - 1)];
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bf16 v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = (bf16)(k0 + s * 32 + g * 8 + j < p.dim ? q[s][j] : 0.0f);
                acc = mma16<bf16>(w[s], __builtin_bit_cast(pi_u32x4, v), acc);
            }
        }
        if (i >= p.T) return;
        bf16 * o = (bf16 *)p.q_lat + ((size_t)i * p.n_head + h) * p.kd + row0 + 4 * g;
#pragma unroll
        for (int k = 0; k < 4; ++k) if (row0 + 4 * g + k < p.kv_rank) o[k] = (bf16)acc[k];
        return;
    }
    b -= n_absorb;
    const int n_rope = (p.n_head * half + kRopePerWg - 1) / kRopePerWg, kinds = n_rope + (p.cache ? 1 : 0) + (r.ids ? 1 : 0), t = b / kinds, what = b % kinds;
    const float * z = p.z + (size_t)t * p.ldz;
    const float2 * cs = (const float2 *)p.cs + (size_t)t * half;
    if (what < n_rope) {                                      // rotated query parts
        float u[kRopePerWg / 256], v[kRopePerWg / 256];
        const int e0 = what * kRopePerWg + tid, last = p.n_head * half - 1;
#pragma unroll
        for (int k = 0; k < kRopePerWg / 256; ++k) {
            const int e = min(e0 + k * 256, last), h = e / half, i = e - h * half;
            u[k] = z[h * hd + p.dim + 2 * i]; v[k] = z[h * hd + p.dim + 2 * i + 1];
        }
#pragma unroll
        for (int k = 0; k < kRopePerWg / 256; ++k) {
            const int e = e0 + k * 256, h = e / half, i = e - h * half;
            if (e > last) continue;
            bf16 * o = (bf16 *)p.q_lat + ((size_t)t * p.n_head + h) * p.kd + p.rank_ld + 2 * i;
            o[0] = (bf16)(u[k] * cs[i].x - v[k] * cs[i].y);
            o[1] = (bf16)(v[k] * cs[i].x + u[k] * cs[i].y);
        }
    } else if (what == n_rope && p.cache) {                        // the token's cell
        const float * c = z + p.n_head * hd;
        bf16 * cell = (bf16 *)p.cache + (size_t)p.cell[t] * p.kd;
        double s = 0.0;
        for (int i = tid; i < p.kv_rank; i += 256) { const float v = c[i]; s += (double)v * (double)v; }
        s = block_sum_f64(s, red);
        const float sc = pi_inv_sqrt((float)(s / p.kv_rank) + p.eps);
        for (int i = tid; i < p.kv_rank; i += 256) cell[i] = (bf16)(c[i] * sc * p.norm_w[i]);
        for (int i = tid; i < half; i += 256) {
            const float u = c[p.kv_rank + 2 * i], v = c[p.kv_rank + 2 * i + 1];
            cell[p.rank_ld + 2 * i] = (bf16)(u * cs[i].x - v * cs[i].y);
            cell[p.rank_ld + 2 * i + 1] = (bf16)(v * cs[i].x + u * cs[i].y);
        }
    } else {                                                  // the token's experts
        route_token(r, t, sm);
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// the parts of a split attention merged (fixed order, the sink in the denominator) and the head's values expanded from the result:
// a workgroup owns 64 value rows of one head, for all tokens of the step
// ---------------------------------------------------------------------------------------------------------------------------------
__host__ __device__ inline size_t value_lds_bytes(int T, int rank_ld, int n_parts) {
    return (size_t)T * (rank_ld + 8) * 2 + sizeof(float) * (((size_t)T * n_parts + 3) / 4 * 4 + 4 * (size_t)rank_ld);
}
__device__ void latent_value(const pi_latent_attn & p, const uint16_t * __restrict__ uv, int vdim, bf16 * __restrict__ att, int ld_att, int h, int rt, unsigned char * smem) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int ld = p.rank_ld + 8;
    bf16 * ol = reinterpret_cast<bf16 *>(smem);               // [T][ld]
    float * f = reinterpret_cast<float *>(ol + p.T * ld);     // [T][n_parts] factor of each part
    float * ws = f + (p.T * p.n_parts + 3) / 4 * 4;           // [4][rank_ld] the waves' sums
    const int row0 = rt * 64 + wave * 16;
    // the value matrix does not depend on the attention: its first fragments are requested ahead of everything else
    const uint16_t * W = uv + ((size_t)h * vdim + min(row0 + i, vdim - 1)) * p.rank_ld + g * 8;
    pi_u32x4 w0[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w0[k] = k * 32 < p.rank_ld ? pi_ld_stream(W + k * 32) : pi_u32x4{0, 0, 0, 0};
    if (p.n_parts == 1) {
        for (int c = tid; c < p.T * (p.rank_ld / 8); c += 256) {
            const int t = c / (p.rank_ld / 8), k = (c % (p.rank_ld / 8)) * 8;
            *reinterpret_cast<pi_u32x4 *>(ol + t * ld + k) = pi_ld16((const uint16_t *)p.out_lat + ((size_t)t * p.n_head + h) * p.rank_ld + k);
        }
    } else {
        const float * ml = p.scratch + (size_t)p.T * p.n_head * p.n_parts * p.rank_ld;
        const float sink = p.sink[h];
        for (int t = wave; t < p.T; t += 4) {                 // a wave per token: n_parts <= 64 lanes
            const float2 v = lane < p.n_parts ? reinterpret_cast<const float2 *>(ml)[((size_t)t * p.n_head + h) * p.n_parts + lane] : make_float2(-INFINITY, 0.0f);
            const float m = fmaxf(pi_wave_max(v.x), sink);
            const float e = v.x == -INFINITY ? 0.0f : expf(v.x - m);
            const float l = pi_wave_sum(e * v.y) + expf(sink - m);
            if (lane < p.n_parts) f[t * p.n_parts + lane] = e / l;
        }
        __syncthreads();
        for (int t = 0; t < p.T; ++t) {                       // a wave takes every fourth part, a lane four columns of a 256-column piece
            const float * a = p.scratch + ((size_t)t * p.n_head + h) * p.n_parts * p.rank_ld;
            for (int c = lane * 4; c < p.rank_ld; c += 256) {
                float4 s = make_float4(0, 0, 0, 0);
                for (int q0 = wave; q0 < p.n_parts; q0 += 32) {
                    float4 v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const float4 *>(a + (size_t)min(q0 + 4 * u, p.n_parts - 1) * p.rank_ld + c);
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const float w = q0 + 4 * u < p.n_parts ? f[t * p.n_parts + q0 + 4 * u] : 0.0f;
                        s.x = fmaf(w, v[u].x, s.x); s.y = fmaf(w, v[u].y, s.y); s.z = fmaf(w, v[u].z, s.z); s.w = fmaf(w, v[u].w, s.w);
                    }
                }
                *reinterpret_cast<float4 *>(ws + wave * p.rank_ld + c) = s;
            }
            __syncthreads();
            for (int c = tid; c < p.rank_ld; c += 256) ol[t * ld + c] = (bf16)(ws[c] + ws[p.rank_ld + c] + ws[2 * p.rank_ld + c] + ws[3 * p.rank_ld + c]);
            __syncthreads();
        }
    }
    __syncthreads();
    if (row0 >= vdim) return;
    const bf16 * x = ol + min(i, p.T - 1) * ld + g * 8;
    pi_f4 acc = pi_f4{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (k * 32 < p.rank_ld) acc = mma16<bf16>(w0[k], *reinterpret_cast<const pi_u32x4 *>(x + k * 32), acc);
    for (int k0 = 256; k0 < p.rank_ld; k0 += 256) {
#pragma unroll
        for (int k = 0; k < 8; ++k) w0[k] = k0 + k * 32 < p.rank_ld ? pi_ld_stream(W + k0 + k * 32) : pi_u32x4{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 8; ++k) if (k0 + k * 32 < p.rank_ld) acc = mma16<bf16>(w0[k], *reinterpret_cast<const pi_u32x4 *>(x + k0 + k * 32), acc);
    }
    if (i >= p.T) return;
    bf16 * o = att + (size_t)i * ld_att + h * vdim + row0 + 4 * g;
#pragma unroll
    for (int k = 0; k < 4; ++k) if (row0 + 4 * g + k < vdim) o[k] = (bf16)acc[k];
}

// ---------------------------------------------------------------------------------------------------------------------------------
// Weight rows streamed past the step's tokens: a wave reads 2 rows x 512 B per load (16 rows x 256 columns in eight), passes them
// through its own LDS buffer into the matrix cores' operand layout (as gemm_t16_lds_kernel does) and multiplies.  Columns beyond the
// end of a row are not read (the last piece of the row is read again) and meet zeros.
// ---------------------------------------------------------------------------------------------------------------------------------
constexpr int kWsStride = 512 + 16;
struct WaveStream {
    unsigned char * tile;
    int lane, i, g, lr, lc;
    __device__ __forceinline__ WaveStream(unsigned char * t) : tile(t), lane(threadIdx.x & 63), i(lane & 15), g(lane >> 4), lr(lane >> 5), lc(lane & 31) {}
    // rows row0 .. row0 + 15 (clamped to rows), columns c0 .. c0 + 255 of a matrix of `cols` (a multiple of 32) columns
    __device__ __forceinline__ void load(pi_u32x4 (&ld)[8], const bf16 * W, size_t ldw, int row0, int rows, int c0, int cols) const {
        const int c = min(c0 + lc * 8, cols - 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) ld[j] = pi_ld_stream(W + (size_t)min(row0 + 2 * j + lr, rows - 1) * ldw + c);
    }
    __device__ __forceinline__ void multiply(const pi_u32x4 (&ld)[8], const pi_u32x4 (&b)[8], pi_f4 & acc) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) *reinterpret_cast<pi_u32x4 *>(tile + (2 * j + lr) * kWsStride + lc * 16) = ld[j];
#pragma unroll
        for (int st = 0; st < 8; ++st) acc = mma16<bf16>(*reinterpret_cast<const pi_u32x4 *>(tile + i * kWsStride + (4 * st + g) * 16), b[st], acc);
    }
};

// The step's distinct experts in LDS: expert[k] in order of first appearance, slot[k][t] = token t's pair with it or -1.
constexpr int kStepPairs = 256, kStepExperts = 2048;
struct StepExperts {
    int expert[kStepPairs], rank[kStepPairs], sred[16];
    int16_t slot[kStepPairs][16];
};
// first: kStepExperts ints of LDS
__device__ int step_experts(StepExperts & s, int * first, const int32_t * __restrict__ ids, int n, int top, int E) {
    const int tid = threadIdx.x, e = tid < n ? ids[tid] : 0;
    for (int k = tid; k < E; k += blockDim.x) first[k] = n;
    for (int k = tid; k < n * 8; k += blockDim.x) reinterpret_cast<int *>(s.slot)[k] = -1;
    __syncthreads();
    if (tid < n) atomicMin(&first[e], tid);
    __syncthreads();
    const int lead = tid < n ? first[e] : -1, own = lead == tid ? 1 : 0;
    int total;
    const int rank = block_exclusive_scan_i32(own, &total, s.sred);
    if (own) { s.expert[rank] = e; s.rank[tid] = rank; }
    __syncthreads();
    if (tid < n) s.slot[s.rank[lead]][tid / top] = (int16_t)tid;
    __syncthreads();
    return total;
}

// ---------------------------------------------------------------------------------------------------------------------------------
// first matrices of the step's experts: workgroup (row tile, pair) works for the pair's expert if no earlier pair has the same one, for
// every token that chose it; act[pair] = weight * relu(z)^2, or (glu: rows of gate and up in turn, ff of both together) weight * clamped GLU (weigh_input:
// the clamped GLU of the weighted rows)
// ---------------------------------------------------------------------------------------------------------------------------------
struct ExpertUp { const bf16 * up; int ff, cols; const bf16 * x_ol; const int32_t * ids; const float * weights; int T, top; bf16 * act; int ld_act; int glu = 0; float limit = 0.0f, gain = 0.0f, one = 1.0f; int weigh_input = 0, streams = 0; };
constexpr int kUpLds = 4 * 16 * kWsStride;
__device__ void expert_up(const ExpertUp & a, int tile, int p, unsigned char * smem) {
    constexpr int NW = 4;
    unsigned char (*tiles)[16 * kWsStride] = reinterpret_cast<unsigned char (*)[16 * kWsStride]>(smem);
    const bf16 * up = a.up, * x_ol = a.x_ol; const int32_t * ids = a.ids;
    const int ff = a.ff, cols = a.cols, T = a.T, top = a.top;
    const int e = ids[p], tid = threadIdx.x, wave = tid >> 6;
    if (T > 1 && __syncthreads_or(tid < p && ids[tid] == e)) return;            // p < 256: checked by the launcher
    const WaveStream ws(tiles[wave]);
    const int row0 = tile * 16, n_ss = (cols + 255) / 256;
    const bf16 * W = up + (size_t)e * ff * cols;
    pi_u32x4 ld[2][8];
    pi_f4 acc = pi_f4{0, 0, 0, 0};
    if (wave < n_ss) ws.load(ld[0], W, cols, row0, ff, wave * 256, cols);
    if (wave + NW < n_ss) ws.load(ld[1], W, cols, row0, ff, (wave + NW) * 256, cols);
    for (int s0 = wave; s0 < n_ss; s0 += 2 * NW) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int ss = s0 + b * NW;
            if (ss < n_ss) {
                pi_u32x4 x[8];
#pragma unroll
                for (int st = 0; st < 8; ++st) x[st] = ss * 256 + st * 32 < cols ? pi_ld16(x_ol + ((size_t)(ss * 8 + st) * 64 + ws.g * 16 + ws.i) * 8) : pi_u32x4{0, 0, 0, 0};
                ws.multiply(ld[b], x, acc);
                if (ss + 2 * NW < n_ss) ws.load(ld[b], W, cols, row0, ff, (ss + 2 * NW) * 256, cols);
            }
        }
    }
    float (*cs)[17] = reinterpret_cast<float (*)[17]>(tiles[wave]);
#pragma unroll
    for (int r = 0; r < 4; ++r) cs[4 * ws.g + r][ws.i] = acc[r];
    __syncthreads();
    if (tid >= 256) return;
    const int rr = tid >> 4, t = tid & 15, row = row0 + rr;
    if (row >= ff || t >= T) return;
    if (a.glu) {
        if (rr & 1) return;
        float g = 0.0f, u = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) { g += reinterpret_cast<float (*)[17]>(tiles[w])[rr][t]; u += reinterpret_cast<float (*)[17]>(tiles[w])[rr + 1][t]; }
        for (int k = 0; k < top; ++k) {
            if (ids[t * top + k] != e) continue;
            const float w = a.weights[t * top + k];
            const float y = a.weigh_input ? clamped_glu(w * g, w * u, a.limit, a.gain, a.one) : w * clamped_glu(g, u, a.limit, a.gain, a.one);
            a.act[(size_t)(t * top + k) * a.ld_act + row / 2] = (bf16)y;
        }
        return;
    }
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += reinterpret_cast<float (*)[17]>(tiles[w])[rr][t];
    v = fmaxf(v, 0.0f);
    for (int k = 0; k < top; ++k)
        if (ids[t * top + k] == e) a.act[(size_t)(t * top + k) * a.ld_act + row] = (bf16)(a.weights[t * top + k] * v * v);
}

// The same for one token: the rows of its experts, one behind the other, are dealt out evenly to `streams` workgroups, two a compute unit; each wave
// takes a quarter of the columns of all rows of its workgroup, its part of the token in registers, two groups of eight loads of 1 KB on
// their way.  Bound by the weights and 4 us ahead of them: which experts they are, then the first rows.  Six experts' 2816 x 4096: 31.3 -> 27 us, 5.1 TB/s
// (in tiles of 16 rows these are 1056 workgroups, of which a unit holds three: two rounds, the second nearly empty).
template <int L>                                        // loads of a row: columns / 2048
__device__ void expert_up_one(const ExpertUp & a, int wg, unsigned char * smem) {
    constexpr int D = 8 / L;                            // rows of a group
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, per_unit = a.glu ? 2 : 1, units = a.top * a.ff / per_unit, per = (units + a.streams - 1) / a.streams;
    const int r0 = wg * per * per_unit, n = min(per * per_unit, a.top * a.ff - r0), rows = per * per_unit;
    if (n <= 0) return;
    float * part = reinterpret_cast<float *>(smem);     // [4][rows]
    const int c0 = wave * (512 * L) + lane * 8;
    float x[L][8];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        const pi_u32x4 v = pi_ld16(a.x_ol + (size_t)(c0 / 8 + 64 * l) * 128);
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[l][2 * e] = __uint_as_float(v[e] << 16); x[l][2 * e + 1] = __uint_as_float(v[e] & 0xFFFF0000u); }
    }
    pi_u32x4 ld[2][D][L];
    auto request = [&](int b, int g) {                  // past the end the last row again, not used
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int r = r0 + min(g * D + d, n - 1), k = r / a.ff;
            const bf16 * w = a.up + ((size_t)a.ids[k] * a.ff + (r - k * a.ff)) * a.cols + c0;
#pragma unroll
            for (int l = 0; l < L; ++l) ld[b][d][l] = pi_ld_stream(w + 512 * l);
        }
    };
    auto multiply = [&](int b, int g) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            float s[2] = {0.0f, 0.0f};
#pragma unroll
            for (int l = 0; l < L; ++l)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[0] = fmaf(__uint_as_float(ld[b][d][l][e] << 16), x[l][2 * e], s[0]);
                    s[1] = fmaf(__uint_as_float(ld[b][d][l][e] & 0xFFFF0000u), x[l][2 * e + 1], s[1]);
                }
            const float t = pi_wave_sum(s[0] + s[1]);
            if (lane == 0 && g * D + d < n) part[wave * rows + g * D + d] = t;
        }
    };
    const int groups = (n + D - 1) / D;
    request(0, 0);
    for (int g = 0; g < groups; g += 2) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            request(b ^ 1, g + b + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(b, g + b);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
    auto sum = [&](int r) { return part[r] + part[rows + r] + part[2 * rows + r] + part[3 * rows + r]; };
    for (int u = tid; u < n / per_unit; u += 256) {
        const int r = r0 + u * per_unit, k = r / a.ff, row = r - k * a.ff;
        const float w = a.weights[k];
        float y;
        if (a.glu) {
            const float g = sum(2 * u), v = sum(2 * u + 1);
            y = a.weigh_input ? clamped_glu(w * g, w * v, a.limit, a.gain, a.one) : w * clamped_glu(g, v, a.limit, a.gain, a.one);
        } else {
            const float v = fmaxf(sum(u), 0.0f);
            y = w * v * v;
        }
        a.act[(size_t)k * a.ld_act + row / per_unit] = (bf16)y;
    }
}
__device__ __forceinline__ void expert_up_any(const ExpertUp & a, int b, int n_tiles, unsigned char * smem) {
    if (!a.streams) expert_up(a, b % n_tiles, b / n_tiles, smem);
    else if (a.cols == 2048) expert_up_one<1>(a, b, smem);
    else if (a.cols == 4096) expert_up_one<2>(a, b, smem);
    else expert_up_one<4>(a, b, smem);
}
// Workgroups of the experts' first matrices.  One token of 2048, 4096 or 8192 columns goes by streams.  Of 2048 columns a group of requests is eight rows and
// a stream asks for them two groups at a time, so its time goes with its rows in sixteens, while a tile of 16 rows is done in one trip and most
// tiles side by side: streams pay from 15 rows each on, where few of the rows asked for are missing.  us, tiles / streams, six experts, by
// rows a stream: 8 8.8 / 9.6, 14 10.1 / 10.3, 16 11.9 / 10.6, 18 12.7 / 14.5, 24 13.6 / 15.3, 28 17.1 / 16.0, 32 18.7 / 16.6, 34 19.4 / 20.2, 38 20.8 /
// 20.6, 48 25.0 / 21.6, 50 25.0 / 25.2, 56 27.7 / 25.8, 66 32.0 / 30.3 (6 x 2816 rows are 34 each).  Experts x rows of 4096 columns: 1 x 32
// 7.2 / 5.0, 4 x 512 9.0 / 8.5, 6 x 2816 30.8 / 25.5; 8192 columns 1 x 32 11.6 / 5.4, 4 x 512 15.2 / 10.7.
inline int up_blocks(ExpertUp & u, int n_tiles) {
    const int per_unit = u.glu ? 2 : 1, units = u.top * u.ff / per_unit, most = 2 * pi::compute_units(), rows = most > 0 ? (units + most - 1) / most * per_unit : 0;
    const int missing = (rows + 15) / 16 * 16 - rows;
    const bool pays = u.cols == 4096 || u.cols == 8192 || (u.cols == 2048 && rows >= 15 && 4 * missing <= rows + 2);
    if (u.T == 1 && most > 0 && pays && rows * 16 <= kUpLds) {
        u.streams = units < most ? units : most;
        return u.streams;
    }
    return n_tiles * u.T * u.top;
}

// both in one launch: the value expansion of the attention branch hides behind the experts' weights
__global__ __launch_bounds__(256) void value_and_up_kernel(pi_latent_attn p, const uint16_t * __restrict__ uv, int vdim, bf16 * __restrict__ att, int ld_att, int n_rt, int n_value,
                                                           ExpertUp u, int n_up_tiles) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int b = blockIdx.x;
    if (b < n_value) latent_value(p, uv, vdim, att, ld_att, b / n_rt, b % n_rt, smem);
    else expert_up_any(u, b - n_value, n_up_tiles, smem);
}

// the merge of a split grouped-query attention (four rows a workgroup) and the gated norm of a linear attention (a token or four heads a
// workgroup) beside the experts' first matrices
__global__ __launch_bounds__(256) void mix_and_up_kernel(pi_gqa_attn p, pi_gate_norm gn, int n_merge, int n_gate, ExpertUp u, int n_up_tiles) {
    extern __shared__ __align__(16) unsigned char smem[];
    int b = blockIdx.x;
    if (b < n_gate) { gate_norm_block<bf16>(gn, b, reinterpret_cast<double *>(smem)); return; }
    b -= n_gate;
    if (b < n_merge) {
        const int r4 = gqa_rows(p.wide) / 4;
        const int n = p.all_values ? p.n_kv * p.n_kv : p.n_kv;
        gqa_merge_row(p, b / r4 / n, b / r4 % n, (b % r4) * 4 + (threadIdx.x >> 6));
        return;
    }
    expert_up_any(u, b - n_merge, n_up_tiles, smem);
}

// ---------------------------------------------------------------------------------------------------------------------------------
// what closes a layer: out[t] = x[t] + (W_o att[t] + sum over the token's experts of W_down[e] act[pair]), 16 or 8 rows a workgroup (or, what
// closes a sublayer in front of its norm: out[t] = alpha x[t] + gate * W att[t]).  The pieces of 256 columns of W_o and of every
// expert of the step form one list that the waves take in turn; with 8 rows a wave takes two of its pieces at a time, one behind the
// other in the tile, so that sums are formed in one order whatever the rows.
// Bound by the weights.  A piece's tokens were once read when its turn came: loads return in order, so each piece also waited for the weights
// requested after it and a wave had one piece in flight instead of two; and 16 rows a workgroup leave half the compute units idle at 2048 rows.
// 16 tokens, 2048 rows, 51 of 64 experts of 1408 (306 MB) and dense layers in turn: 65.7 us a layer, 56 with 8 rows and both requested
// together, 53 with the requests free of branches.
// ---------------------------------------------------------------------------------------------------------------------------------
template <int NW, int RT>      // waves, rows a workgroup
__global__ __launch_bounds__(64 * NW) void layer_out_step_kernel(pi_layer_out a) {
    constexpr int COLS = 256, NX = COLS / 32, LR = COLS / 8, PITCH = COLS * 2 + 16;      // columns of a piece, its steps of 32, lanes of a row, bytes of a staged row
    constexpr int NP = 16 / RT, NL = 8 / NP;           // pieces a turn (their rows together fill the tile of 16), loads of a piece
    __shared__ __align__(16) unsigned char tiles[NW][16 * PITCH];
    __shared__ StepExperts se;
    __shared__ int first[kStepExperts];
    // (eight waves: the workgroup's LDS exceeds half a compute unit's, so that no two share one while others idle)
    static_assert(NW < 8 || sizeof(tiles) + sizeof(se) + sizeof(first) > 80 * 1024, "one workgroup per compute unit");
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * RT, n_o = a.wo ? (a.ld_att + COLS - 1) / COLS : 0, n_e = a.ids ? (a.ld_act + COLS - 1) / COLS : 1;
    const int tok = min(i, a.T - 1);
    pi_u32x4 ld[2][8], x[2][NP * NX];
    int left[2][NP];                                   // columns of a piece and behind it; 0: the token has no part in it
    pi_f4 acc = pi_f4{0, 0, 0, 0};
    // a piece's weights and its tokens' values are requested together, two turns ahead and without branches (past the end: the last columns again)
    auto request_piece = [&](pi_u32x4 * l, pi_u32x4 * v, int & rest, int ss) {
        const bool att = ss < n_o;
        const int k = att ? 0 : (ss - n_o) / n_e, c = (att ? ss : (ss - n_o) % n_e) * COLS, cols = att ? a.ld_att : a.ld_act;
        const bf16 * w = att ? (const bf16 *)a.wo : (const bf16 *)a.down + (size_t)se.expert[k] * a.rows * a.ld_act;
        const int at = min(c + (lane % LR) * 8, cols - 8);
#pragma unroll
        for (int j = 0; j < NL; ++j) l[j] = pi_ld_stream(w + (size_t)min(row0 + 2 * j + lane / LR, a.rows - 1) * cols + at);
        const int pair = att ? tok : se.slot[k][i];
        const bf16 * xp = (att ? (const bf16 *)a.att : (const bf16 *)a.act) + (size_t)max(pair, 0) * cols;
#pragma unroll
        for (int st = 0; st < NX; ++st) v[st] = pi_ld16(xp + min(c + st * 32, cols - 32) + g * 8);
        rest = pair >= 0 ? cols - c : 0;
    };
    // turn t of this wave's pieces wave, wave + NW, ..: pieces t NP .. of them, in this order, as far as `upto` goes
    auto piece_of = [&](int t, int p) { return wave + (t * NP + p) * NW; };
    auto request = [&](int b, int t, int from, int upto) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
            if (piece_of(t, p) >= from && piece_of(t, p) < upto) request_piece(&ld[b][p * NL], &x[b][p * NX], left[b][p], piece_of(t, p));
    };
    // the attention's pieces are requested before the experts are known
    request(0, 0, 0, n_o);
    request(1, 1, 0, n_o);
    const int n_exp = a.ids ? step_experts(se, first, a.ids, a.T * a.top, a.top, a.n_expert) : 0, n_ss = n_o + n_exp * n_e;
    const int m = wave < n_ss ? (n_ss - wave + NW - 1) / NW : 0, whole = m / NP;           // this wave's pieces; whole turns of them
    request(0, 0, n_o, n_ss);
    request(1, 1, n_o, n_ss);
    auto multiply = [&](int b, int n) {                // n: pieces of the turn
#pragma unroll
        for (int j = 0; j < 8; ++j) *reinterpret_cast<pi_u32x4 *>(tiles[wave] + (2 * j + lane / LR) * PITCH + (lane % LR) * 16) = ld[b][j];
#pragma unroll
        for (int p = 0; p < NP; ++p)
            if (p < n) {
#pragma unroll
                for (int st = 0; st < NX; ++st)
                    acc = mma16<bf16>(*reinterpret_cast<const pi_u32x4 *>(tiles[wave] + (p * RT + i % RT) * PITCH + (4 * st + g) * 16),
                                      st * 32 < left[b][p] ? x[b][p * NX + st] : pi_u32x4{0, 0, 0, 0}, acc);
            }
    };
    // (no branch around a request while whole turns are left for both buffers: what a wait leaves in flight is then known when it is compiled)
    int t = 0;
    for (; t + 4 <= whole; t += 2)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            multiply(b, NP);
#pragma unroll
            for (int p = 0; p < NP; ++p) request_piece(&ld[b][p * NL], &x[b][p * NX], left[b][p], piece_of(t + 2 + b, p));
        }
    // up to four turns, the last of which may be short of a piece
    const int turns = (m + NP - 1) / NP - t;
#pragma unroll
    for (int b = 0; b < 2; ++b)
        if (b < turns) {
            multiply(b, m - (t + b) * NP);
            if (b + 2 < turns) request(b, t + b + 2, 0, n_ss);
        }
#pragma unroll
    for (int b = 0; b < 2; ++b)
        if (b + 2 < turns) multiply(b, m - (t + b + 2) * NP);
    float (*cs)[17] = reinterpret_cast<float (*)[17]>(tiles[wave]);
#pragma unroll
    for (int r = 0; r < 4; ++r) if (4 * g + r < RT) cs[4 * g + r][i] = acc[r];
    __syncthreads();
    if (tid >= 16 * RT) return;
    const int tk = tid / RT, row = row0 + tid % RT;
    if (row >= a.rows || tk >= a.T) return;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += reinterpret_cast<float (*)[17]>(tiles[w])[tid % RT][tk];
    if (a.gate_z) v *= sigmoid_f32(a.gate_z[(size_t)tk * a.ld_gate + a.off_gate + row] + a.gate_b[row]);
    const float x0 = a.x ? a.x[(size_t)tk * a.rows + row] : 0.0f;
    v += a.scaled ? a.alpha * x0 : x0;
    a.out[(size_t)tk * a.rows + row] = v;
    if (a.keep) a.keep[(size_t)tk * a.rows + row] = v;
}

// The same for one token: `per` rows a workgroup, one workgroup a compute unit.  W_o's columns and those of the token's experts are one row of pieces of 8; a
// thread has every 512th of them for all of the rows, with the token's values there in registers.
// Bound by the weights and the launch: six experts of 1408 to 4096 rows 17.5 -> 14.8 us (4.7 TB/s), 4096 x 4096 alone 9.3 both.
constexpr int kOneRows = 64, kOnePieces = 6;            // most rows of a workgroup, pieces of a thread
template <int J>
__global__ __launch_bounds__(512) void layer_out_one_kernel(pi_layer_out a, int per) {
    constexpr int D = J == 1 ? 8 : J == 2 ? 4 : J == 3 ? 3 : 2;      // rows of a group: two groups are on their way
    __shared__ float part[8][kOneRows];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, row0 = blockIdx.x * per, n = min(per, a.rows - row0);
    const int n_att = a.wo ? a.ld_att / 8 : 0, n_act = a.ids ? a.ld_act / 8 : 1, total = n_att + (a.ids ? a.top * n_act : 0);
    const bf16 * w[J];
    int ldw[J];
    float x[J][8];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int q = min(tid + 512 * j, total - 1);    // (past the end the last piece again, not used)
        const bool att = q < n_att;
        const int k = att ? 0 : (q - n_att) / n_act, c = (att ? q : (q - n_att) % n_act) * 8;
        ldw[j] = att ? a.ld_att : a.ld_act;
        w[j] = (att ? (const bf16 *)a.wo : (const bf16 *)a.down + (size_t)a.ids[k] * a.rows * a.ld_act) + (size_t)row0 * ldw[j] + c;
        const pi_u32x4 v = pi_ld16((att ? (const bf16 *)a.att : (const bf16 *)a.act + (size_t)k * a.ld_act) + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[j][2 * e] = __uint_as_float(v[e] << 16); x[j][2 * e + 1] = __uint_as_float(v[e] & 0xFFFF0000u); }
    }
    const bool last = tid + 512 * (J - 1) < total;      // the others hold a piece less (not one times zero: a weight may be infinite)
    pi_u32x4 ld[2][D][J];
    auto request = [&](int b, int g) {                  // past the end the last row again, not used
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
            for (int j = 0; j < J; ++j) ld[b][d][j] = pi_ld_stream(w[j] + (size_t)min(g * D + d, n - 1) * ldw[j]);
    };
    auto multiply = [&](int b, int g) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            float s[2] = {0.0f, 0.0f}, less = 0.0f;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if (j == J - 1) less = s[0] + s[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[0] = fmaf(__uint_as_float(ld[b][d][j][e] << 16), x[j][2 * e], s[0]);
                    s[1] = fmaf(__uint_as_float(ld[b][d][j][e] & 0xFFFF0000u), x[j][2 * e + 1], s[1]);
                }
            }
            const float t = pi_wave_sum(last ? s[0] + s[1] : less);
            if (lane == 0 && g * D + d < n) part[wave][g * D + d] = t;
        }
    };
    const int groups = (n + D - 1) / D;
    request(0, 0);
    for (int g = 0; g < groups; g += 2) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            request(b ^ 1, g + b + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(b, g + b);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
    if (tid >= n) return;
    const int row = row0 + tid;
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) v += part[k][tid];
    if (a.gate_z) v *= sigmoid_f32(a.gate_z[a.off_gate + row] + a.gate_b[row]);
    const float x0 = a.x ? a.x[row] : 0.0f;
    v += a.scaled ? a.alpha * x0 : x0;
    a.out[row] = v;
    if (a.keep) a.keep[row] = v;
}

}  // namespace

extern "C" {

int pi_k_layer_step_supported(int T, int n_expert, int n_top) { return T >= 1 && T <= kBtMaxT && n_expert <= kStepExperts && T * n_top <= kStepPairs; }

int pi_k_latent_step(const pi_latent_prep * p, const void * uk_t, const float * z_router, int n_expert, int n_top, int n_group, int n_keep, const float * bias,
                     int32_t * ids, float * weights, pi_stream_t stream) {
    if (!p || !p->z || !p->q_lat || !p->cs || !uk_t || p->T <= 0 || p->T > kBtMaxT || p->n_head <= 0 || p->dim <= 0 || p->dim_ld % 32 || p->dim_ld < p->dim || p->rot_dim <= 0 ||
        p->rot_dim % 2 || p->kv_rank <= 0 || p->rank_ld < p->kv_rank || p->kd < p->rank_ld + p->rot_dim || (p->cache && (!p->cell || !p->norm_w)) ||
        p->ldz < p->n_head * (p->dim + p->rot_dim) + (p->cache ? p->kv_rank + p->rot_dim : 0))
        return pi::fail(PI_E_ARG, "pi_k_latent_step: bad arguments");
    if (ids && (!z_router || !bias || !weights || n_expert <= 0 || n_expert > kStepExperts || n_group <= 0 || n_expert % n_group || n_keep <= 0 || n_keep > n_group || n_top <= 0 ||
                n_top > n_keep * (n_expert / n_group)))
        return pi::fail(PI_E_ARG, "pi_k_latent_step: bad routing arguments");
    const int n_absorb = p->n_head * ((p->kv_rank + 63) / 64), kinds = (p->n_head * (p->rot_dim / 2) + kRopePerWg - 1) / kRopePerWg + (p->cache ? 1 : 0) + (ids ? 1 : 0);
    hipLaunchKernelGGL(latent_step_kernel, dim3(n_absorb + p->T * kinds), dim3(256), ids ? route_lds_bytes(n_expert, n_group, n_top) : 0, (hipStream_t)stream, *p, (const uint16_t *)uk_t,
                       RouteArgs{z_router, n_expert, n_top, n_group, n_keep, bias, ids, weights}, n_absorb);
    return pi::check_launch("pi_k_latent_step");
}

int pi_k_value_up_step(const pi_latent_attn * p, const void * uv, int vdim, void * att, int ld_att, const void * up, int n_expert, int ff, int cols, const void * x_ol,
                       const int32_t * ids, const float * weights, int top, void * act, int ld_act, pi_stream_t stream) {
    if (!p || !uv || !att || p->T <= 0 || p->T > kBtMaxT || p->n_head <= 0 || vdim <= 0 || p->rank_ld <= 0 || p->rank_ld % 64 || p->rank_ld > 1024 || ld_att < p->n_head * vdim || !p->sink ||
        p->n_parts <= 0 || p->n_parts > 64 || (p->n_parts == 1 ? !p->out_lat : !p->scratch))
        return pi::fail(PI_E_ARG, "pi_k_value_up_step: bad arguments");
    if (ids && (!up || !x_ol || !weights || !act || n_expert <= 0 || ff <= 0 || cols <= 0 || cols % 32 || top <= 0 || p->T * top > kStepPairs || ld_act < ff))
        return pi::fail(PI_E_ARG, "pi_k_value_up_step: bad expert arguments");
    const int n_rt = (vdim + 63) / 64, n_value = p->n_head * n_rt, n_up_tiles = ids ? (ff + 15) / 16 : 1;
    ExpertUp u{(const bf16 *)up, ff, cols, (const bf16 *)x_ol, ids, weights, p->T, top, (bf16 *)act, ld_act};
    const int n_up = ids ? up_blocks(u, n_up_tiles) : 0;
    size_t lds = value_lds_bytes(p->T, p->rank_ld, p->n_parts);
    if (ids && lds < (size_t)kUpLds) lds = kUpLds;
    static bool raised = false;
    if (!raised) { PI_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&value_and_up_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024)); raised = true; }
    hipLaunchKernelGGL(value_and_up_kernel, dim3(n_value + n_up), dim3(256), lds, (hipStream_t)stream, *p, (const uint16_t *)uv, vdim, (bf16 *)att, ld_att, n_rt, n_value, u, n_up_tiles);
    return pi::check_launch("pi_k_value_up_step");
}

int pi_k_mix_up_step(const pi_gqa_attn * attn, const pi_gate_norm * gate, const void * up, int n_expert, int ff, int cols, float limit, float gain, const void * x_ol, int T,
                     const int32_t * ids, const float * weights, int top, void * act, int ld_act, pi_stream_t stream) {
    const pi_gqa_attn p = attn ? *attn : pi_gqa_attn{};
    const pi_gate_norm g = gate ? *gate : pi_gate_norm{};
    if (T <= 0 || T > kBtMaxT || (attn && (!p.att || !p.scratch || !p.work || p.n_parts <= 1 || p.n_parts > 64 || p.n_work <= 0 || p.n_kv <= 0 || p.n_head % p.n_kv || p.vdim <= 0 || p.hd < p.vdim)) ||
        (gate && (!gate_norm_ok(g) || g.T != T)))
        return pi::fail(PI_E_ARG, "pi_k_mix_up_step: bad arguments");
    if (ids && (!up || !x_ol || !weights || !act || n_expert <= 0 || ff <= 0 || cols <= 0 || cols % 32 || top <= 0 || T * top > kStepPairs || ld_act < ff))
        return pi::fail(PI_E_ARG, "pi_k_mix_up_step: bad expert arguments");
    const int n_merge = attn ? p.n_work * p.n_kv * (p.all_values ? p.n_kv : 1) * (gqa_rows(p.wide) / 4) : 0, n_gate = gate ? gate_norm_blocks(g) : 0, n_up_tiles = ids ? (2 * ff + 15) / 16 : 1;
    ExpertUp u{(const bf16 *)up, 2 * ff, cols, (const bf16 *)x_ol, ids, weights, T, top, (bf16 *)act, ld_act};
    u.glu = 1; u.limit = limit; u.gain = gain;
    const int n_up = ids ? up_blocks(u, n_up_tiles) : 0;
    if (n_merge + n_gate + n_up == 0) return PI_OK;
    hipLaunchKernelGGL(mix_and_up_kernel, dim3(n_merge + n_gate + n_up), dim3(256), ids ? kUpLds : 256, (hipStream_t)stream, p, g, n_merge, n_gate, u, n_up_tiles);
    return pi::check_launch("pi_k_mix_up_step");
}

int pi_k_expert_up_step(const void * up, int n_expert, int ff, int cols, float limit, float gain, int plain_up, int weigh_input, const void * x_ol, int T, const int32_t * ids,
                        const float * weights, int top, void * act, int ld_act, pi_stream_t stream) {
    if (!up || !x_ol || !ids || !weights || !act || T <= 0 || T > kBtMaxT || n_expert <= 0 || ff <= 0 || cols <= 0 || cols % 32 || top <= 0 || T * top > kStepPairs || ld_act < ff)
        return pi::fail(PI_E_ARG, "pi_k_expert_up_step: bad arguments");
    ExpertUp u{(const bf16 *)up, 2 * ff, cols, (const bf16 *)x_ol, ids, weights, T, top, (bf16 *)act, ld_act};
    u.glu = 1; u.limit = limit; u.gain = gain; u.one = plain_up ? 0.0f : 1.0f; u.weigh_input = weigh_input;
    const int tiles = (2 * ff + 15) / 16, blocks = up_blocks(u, tiles);
    hipLaunchKernelGGL(mix_and_up_kernel, dim3(blocks), dim3(256), kUpLds, (hipStream_t)stream, pi_gqa_attn{}, pi_gate_norm{}, 0, 0, u, tiles);
    return pi::check_launch("pi_k_expert_up_step");
}

}  // extern "C"

namespace pi {
int expert_relu2_step(const void * up, int n_expert, int ff, int cols, const void * x_ol, int T, const int32_t * ids, const float * weights, int top, void * act, int ld_act,
                      pi_stream_t stream) {
    if (!up || !x_ol || !ids || !weights || !act || T <= 0 || T > kBtMaxT || n_expert <= 0 || ff <= 0 || cols <= 0 || cols % 32 || top <= 0 || T * top > kStepPairs || ld_act < ff)
        return fail(PI_E_ARG, "expert_relu2_step: bad arguments");
    const int tiles = (ff + 15) / 16;
    ExpertUp u{(const bf16 *)up, ff, cols, (const bf16 *)x_ol, ids, weights, T, top, (bf16 *)act, ld_act};
    const int blocks = up_blocks(u, tiles);
    hipLaunchKernelGGL(mix_and_up_kernel, dim3(blocks), dim3(256), kUpLds, (hipStream_t)stream, pi_gqa_attn{}, pi_gate_norm{}, 0, 0, u, tiles);
    return check_launch("expert_relu2_step");
}
}  // namespace pi

extern "C" {

int pi_k_layer_out_step(const pi_layer_out * a, pi_stream_t stream) {
    if (!a || (a->wo ? !a->att || a->ld_att <= 0 || a->ld_att % 32 : !a->ids) || !a->out || (a->gate_z && (!a->gate_b || a->off_gate < 0 || a->off_gate + a->rows > a->ld_gate)) || a->rows <= 0 || a->T <= 0 || a->T > kBtMaxT ||
        (a->ids && (!a->down || !a->act || a->ld_act <= 0 || a->ld_act % 32 || a->top <= 0 || a->T * a->top > kStepPairs || a->n_expert <= 0 || a->n_expert > kStepExperts)))
        return pi::fail(PI_E_ARG, "pi_k_layer_out_step: bad arguments");
    // eight waves a workgroup when every workgroup has a compute unit to itself, four (and several workgroups a unit) beyond
    // Eight rows a workgroup (half of each matrix tile repeats them) while 16 would leave half the units without one.
    const int n = (a->rows + 15) / 16, cus = pi::compute_units();
    // One token goes by streams of rows from a second piece for some threads on: up to 4096 columns (W_o's and the experts' together) part of a workgroup has
    // none, and the tiles are the faster ones where the matrix is small.  With experts, which the tiles look up first, streams pay from there down
    // to 3072 columns; with 4096 for more than 2048 rows, except where the tiles are two for every unit; and with more rows than that from 2048 columns on.
    // us, tiles / streams: 2048 x 2048 4.8 / 5.9, 2048 x 4096 7.0 / 7.4, 4096 x 1024 4.4 / 5.7, 4096 x 3072 7.2 / 7.5, 8192 x 4096 15.7 / 16.4; 2048 x (2048 + 2 x
    // 256) 6.2 / 6.3; 2048 x (2048 + 2 x 704) 6.9 / 6.7, 4096 x 4096 9.8 / 8.5, 12288 x 2048 15.0 / 12.8, 1024 x 6144 7.2 / 6.3, 2048 x 6144 8.3 / 7.2, 5120 x
    // 12288 29.2 / 21.9.
    const int columns = (a->wo ? a->ld_att : 0) + (a->ids ? a->top * a->ld_act : 0);
    const int pieces = (columns / 8 + 511) / 512, per = cus > 0 ? (a->rows + cus - 1) / cus : kOneRows + 1;
    const bool streams = columns > (a->ids ? 3072 : 4096) || (columns == 4096 && a->rows > 2048 && n != 2 * cus) || (columns >= 2048 && n > 2 * cus);
    if (a->T == 1 && streams && pieces <= kOnePieces && per <= kOneRows) {
        const dim3 grid((a->rows + per - 1) / per);
        switch (pieces) {
            case 1: hipLaunchKernelGGL(layer_out_one_kernel<1>, grid, dim3(512), 0, (hipStream_t)stream, *a, per); break;
            case 2: hipLaunchKernelGGL(layer_out_one_kernel<2>, grid, dim3(512), 0, (hipStream_t)stream, *a, per); break;
            case 3: hipLaunchKernelGGL(layer_out_one_kernel<3>, grid, dim3(512), 0, (hipStream_t)stream, *a, per); break;
            case 4: hipLaunchKernelGGL(layer_out_one_kernel<4>, grid, dim3(512), 0, (hipStream_t)stream, *a, per); break;
            case 5: hipLaunchKernelGGL(layer_out_one_kernel<5>, grid, dim3(512), 0, (hipStream_t)stream, *a, per); break;
            default: hipLaunchKernelGGL(layer_out_one_kernel<6>, grid, dim3(512), 0, (hipStream_t)stream, *a, per);
        }
        return pi::check_launch("pi_k_layer_out_step");
    }
    if (2 * n <= cus) hipLaunchKernelGGL((layer_out_step_kernel<8, 8>), dim3((a->rows + 7) / 8), dim3(512), 0, (hipStream_t)stream, *a);
    else if (n <= cus) hipLaunchKernelGGL((layer_out_step_kernel<8, 16>), dim3(n), dim3(512), 0, (hipStream_t)stream, *a);
    else hipLaunchKernelGGL((layer_out_step_kernel<4, 16>), dim3(n), dim3(256), 0, (hipStream_t)stream, *a);
    return pi::check_launch("pi_k_layer_out_step");
}

}  // extern "C"
