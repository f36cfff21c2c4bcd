// Layers with a norm before and after every sublayer: norms in groups, the sum that closes a sublayer together with the norm in front of the next
// one, and the norm with a causal convolution over time behind it.
#include "layer_types.hpp"
#include "mixers.hpp"
#include "route.hpp"

namespace {

constexpr int kNormMaxCols = 32768;

// scale[r * groups + g] = 1 / root mean square of group g of row r, for `rows` rows (at(r): their first value, in global memory or LDS).  part:
// group_parts floats.  Every (row, group) falls into equal pieces so that all waves have one.
__host__ __device__ inline int group_parts(int rows, int groups, int waves) { const int n = rows * groups; return n >= waves ? n : (waves + n - 1) / n * n; }
template <typename AT>
__device__ void group_scales(float * part, float * scale, int rows, int groups, int cols, float eps, AT && at) {
    const int nw = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, size = cols / groups, n = rows * groups, segs = group_parts(rows, groups, nw) / n;
    const int seg = ((size + segs - 1) / segs + 3) / 4 * 4;
    const bool quads = (size & 3) == 0;
    for (int task = wave; task < n * segs; task += nw) {
        const int rg = task / segs, s = task % segs, r = rg / groups, lo = min(s * seg, size), hi = min(lo + seg, size);
        const float * p = at(r) + (rg % groups) * size;
        float sum = 0.0f;
        if (quads) {
#pragma unroll 4
            for (int c = lo + lane * 4; c < hi; c += 256) {
                const float4 v = *reinterpret_cast<const float4 *>(p + c);
                sum = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, sum))));
            }
        } else {
            for (int c = lo + lane; c < hi; c += 64) sum = fmaf(p[c], p[c], sum);
        }
        sum = pi_wave_sum(sum);
        if (lane == 0) part[task] = sum;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        float s = 0.0f;
        for (int k = 0; k < segs; ++k) s += part[i * segs + k];
        scale[i] = pi_inv_sqrt(s / (float)size + eps);
    }
    __syncthreads();
}

// one token a workgroup, its row in LDS
template <typename ST>
__global__ void sum_norm_kernel(pi_sum_norm p) {
    extern __shared__ __align__(16) float sm[];
    const int t = blockIdx.x, tid = threadIdx.x, nt = blockDim.x, size = p.cols / p.groups;
    float * buf = sm, * scale = sm + (p.cols + 3) / 4 * 4, * part = scale + p.groups;
    const size_t base = (size_t)(p.rows ? p.rows[t] : t) * p.cols;
    const bool quads = (p.cols & 3) == 0 && (size & 3) == 0;      // four columns lie in one group
    if (p.w) {
        const float * mix = p.mix ? p.mix + base : nullptr;
        if (quads) {
            struct alignas(4 * sizeof(ST)) Quad { ST v[4]; };
            for (int c = tid * 4; c < p.cols; c += nt * 4) {
                float4 v = mix ? *reinterpret_cast<const float4 *>(mix + c) : make_float4(0, 0, 0, 0);
                if (!mix) for (int k = 0; k < p.top; ++k) {
                    const Quad q = *reinterpret_cast<const Quad *>((const ST *)p.y + (size_t)p.inv[t * p.top + k] * p.cols + c);
                    const float w = p.y_w ? p.y_w[t * p.top + k] : 1.0f;
                    v.x = fmaf(w, from_st(q.v[0]), v.x); v.y = fmaf(w, from_st(q.v[1]), v.y); v.z = fmaf(w, from_st(q.v[2]), v.z); v.w = fmaf(w, from_st(q.v[3]), v.w);
                }
                *reinterpret_cast<float4 *>(buf + c) = v;
            }
        } else {
            for (int c = tid; c < p.cols; c += nt) {
                float v = mix ? mix[c] : 0.0f;
                if (!mix) for (int k = 0; k < p.top; ++k) v = fmaf(p.y_w ? p.y_w[t * p.top + k] : 1.0f, from_st(((const ST *)p.y)[(size_t)p.inv[t * p.top + k] * p.cols + c]), v);
                buf[c] = v;
            }
        }
        __syncthreads();
        group_scales(part, scale, 1, p.groups, p.cols, p.eps, [&](int) { return buf; });
        float * x = p.x + base, * keep = p.keep ? p.keep + base : nullptr;
        if (quads) {
            for (int c = tid * 4; c < p.cols; c += nt * 4) {
                const float f = p.mult * scale[c / size];
                const float4 b = *reinterpret_cast<const float4 *>(buf + c), w = *reinterpret_cast<const float4 *>(p.w + c), o = *reinterpret_cast<const float4 *>(x + c);
                const float4 v = make_float4(fmaf(f * b.x, w.x, o.x), fmaf(f * b.y, w.y, o.y), fmaf(f * b.z, w.z, o.z), fmaf(f * b.w, w.w, o.w));
                *reinterpret_cast<float4 *>(x + c) = v;
                if (keep) *reinterpret_cast<float4 *>(keep + c) = v;
                *reinterpret_cast<float4 *>(buf + c) = v;
            }
        } else {
            for (int c = tid; c < p.cols; c += nt) {
                const float v = fmaf(p.mult * scale[c / size] * buf[c], p.w[c], x[c]);
                x[c] = v;
                if (keep) keep[c] = v;
                buf[c] = v;
            }
        }
    } else {
        for (int c = tid; c < p.cols; c += nt) buf[c] = p.x[base + c];
    }
    if (!p.h) return;
    __syncthreads();
    group_scales(part, scale, 1, p.groups, p.cols, p.eps, [&](int) { return buf; });
    ST * h = (ST *)p.h;
    auto at = [&](int c) -> size_t { return p.ol ? pi_ol_index(t, c) : (size_t)t * p.ld + c; };
    if (quads && (p.ld & 3) == 0) {                    // (four columns from a multiple of four on lie together in both layouts)
        for (int c = tid * 4; c < p.cols; c += nt * 4) {
            const float f = scale[c / size];
            const float4 b = *reinterpret_cast<const float4 *>(buf + c), w = *reinterpret_cast<const float4 *>(p.w_next + c);
            const float v[4] = {f * b.x * w.x, f * b.y * w.y, f * b.z * w.z, f * b.w * w.w};
            store4(h + at(c), v, true, 4);
        }
    } else {
        for (int c = tid; c < p.cols; c += nt) h[at(c)] = to_st<ST>(scale[c / size] * buf[c] * p.w_next[c]);
    }
}

// The same for groups of whole waves: a group of a token's a workgroup, 256 NQ columns a wave in registers.  Bound by latency and by what one unit
// can read: nothing of a group depends on another, and a token's 64 KB or more are some 3 us for one unit alone.  Everything a group needs is
// requested at once, where the kernel above goes to memory three times in a row (the sum, x and the weight behind its norm, the next weight).  4096 columns in
// 8 groups, one token, us: sum and next norm 6.2 -> 4.0, sum alone 4.6 -> 3.3.  Sums in the same order.
template <typename ST, int NQ>
__global__ __launch_bounds__(1024) void sum_norm_quads_kernel(pi_sum_norm p) {
    struct alignas(4 * sizeof(ST)) Quad { ST v[4]; };
    __shared__ float part[2][16];
    const int t = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6, size = p.cols / p.groups, c0 = (int)blockIdx.y * size;
    const size_t base = (size_t)(p.rows ? p.rows[t] : t) * p.cols;
    const auto col = [&](int q) { return c0 + (wave * NQ + q) * 256 + lane * 4; };
    const auto quad = [&](const float * v, int q) { return *reinterpret_cast<const float4 *>(v + col(q)); };
    float4 x[NQ], b[NQ], w[NQ], next[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        if (p.mix) b[q] = quad(p.mix + base, q);
        x[q] = quad(p.x + base, q);
        if (p.w) w[q] = quad(p.w, q);
        if (p.h) next[q] = quad(p.w_next, q);
    }
    // 1 / root mean square of the group
    const auto scaled = [&](const float4 (&v)[NQ], float * sums) -> float {
        float sum = 0.0f, s = 0.0f;
#pragma unroll
        for (int q = 0; q < NQ; ++q) sum = fmaf(v[q].x, v[q].x, fmaf(v[q].y, v[q].y, fmaf(v[q].z, v[q].z, fmaf(v[q].w, v[q].w, sum))));
        sum = pi_wave_sum(sum);
        if (lane == 0) sums[wave] = sum;
        __syncthreads();
        for (int k = 0; k < waves; ++k) s += sums[k];
        return pi_inv_sqrt(s / (float)size + p.eps);
    };
    if (p.w) {
        if (!p.mix) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) b[q] = make_float4(0, 0, 0, 0);
            for (int k = 0; k < p.top; ++k) {
                const ST * y = (const ST *)p.y + (size_t)p.inv[t * p.top + k] * p.cols;
                const float f = p.y_w ? p.y_w[t * p.top + k] : 1.0f;
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    const Quad r = *reinterpret_cast<const Quad *>(y + col(q));
                    b[q].x = fmaf(f, from_st(r.v[0]), b[q].x); b[q].y = fmaf(f, from_st(r.v[1]), b[q].y); b[q].z = fmaf(f, from_st(r.v[2]), b[q].z); b[q].w = fmaf(f, from_st(r.v[3]), b[q].w);
                }
            }
        }
        const float f = p.mult * scaled(b, part[0]);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            x[q] = make_float4(fmaf(f * b[q].x, w[q].x, x[q].x), fmaf(f * b[q].y, w[q].y, x[q].y), fmaf(f * b[q].z, w[q].z, x[q].z), fmaf(f * b[q].w, w[q].w, x[q].w));
            *reinterpret_cast<float4 *>(p.x + base + col(q)) = x[q];
            if (p.keep) *reinterpret_cast<float4 *>(p.keep + base + col(q)) = x[q];
        }
    }
    if (!p.h) return;
    const float f = scaled(x, part[1]);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const float v[4] = {f * x[q].x * next[q].x, f * x[q].y * next[q].y, f * x[q].z * next[q].z, f * x[q].w * next[q].w};
        store4((ST *)p.h + (p.ol ? pi_ol_index(t, col(q)) : (size_t)t * p.ld + col(q)), v, true, 4);
    }
}
// groups of up to 16 waves of 256, 512 or 1024 columns
template <typename ST> bool launch_sum_quads(const pi_sum_norm & p, hipStream_t st) {
    const int size = p.cols / p.groups, nq = size <= 4096 ? 1 : size <= 8192 ? 2 : 4, per = 256 * nq;
    if (size > 16384 || size % per || (p.h && p.ld % 4)) return false;
    const dim3 grid(p.T, p.groups), block(size / per * 64);
    if (nq == 1) hipLaunchKernelGGL((sum_norm_quads_kernel<ST, 1>), grid, block, 0, st, p);
    else if (nq == 2) hipLaunchKernelGGL((sum_norm_quads_kernel<ST, 2>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((sum_norm_quads_kernel<ST, 4>), grid, block, 0, st, p);
    return true;
}

// The same for steps of up to 16 tokens, with the expert choice that reads the normed row: every group's workgroup multiplies its 512 M columns with the
// router's, and the last of a token's to arrive adds the groups' sums in order and chooses.  Bound by latency: the router's rows (64 KB a
// workgroup, 2 us for one unit) travel while the norms are formed, where a product of four workgroups with 128 KB each and the choice were
// launches of their own.  4096 columns in 8 groups, 64 experts, one token: 4.0 + 5.6 + 3.9 -> 7.4 us.  Norms as above; the products in fp32 of the
// row in bf16, as before.
constexpr int kSrWaves = 8, kSrRows = 8, kSrExperts = 256, kSrGroups = 32;
struct SumRoute { const bf16 * router; int ld, E, top; int32_t * ids; float * weights, * sums; unsigned int * arrived; };
template <int M>
__global__ __launch_bounds__(64 * kSrWaves) void sum_norm_route_kernel(pi_sum_norm p, SumRoute r) {
    constexpr int SIZE = 512 * M, NW = SIZE / 256;                  // waves that form the norms
    __shared__ float part[2][NW];
    __shared__ __align__(16) bf16 hs[SIZE];
    __shared__ __align__(16) float z[kSrExperts], sm[3 * kSrExperts];
    __shared__ bool last;
    const int t = blockIdx.x, g = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c0 = g * SIZE, col = c0 + wave * 256 + lane * 4;
    const bool mine = wave < NW;
    const size_t base = (size_t)t * p.cols;
    float4 x{}, b{}, w{}, next{};
    if (mine) {
        b = *reinterpret_cast<const float4 *>(p.mix + base + col); x = *reinterpret_cast<const float4 *>(p.x + base + col);
        w = *reinterpret_cast<const float4 *>(p.w + col); next = *reinterpret_cast<const float4 *>(p.w_next + col);
    }
    pi_u32x4 ld[kSrRows][M];
    const auto rows = [&](int e0) {                                 // experts e0 + wave, e0 + wave + kSrWaves, ..
#pragma unroll
        for (int k = 0; k < kSrRows; ++k)
#pragma unroll
            for (int m = 0; m < M; ++m) ld[k][m] = pi_ld16(r.router + (size_t)min(e0 + wave + k * kSrWaves, r.E - 1) * r.ld + c0 + m * 512 + lane * 8);
    };
    rows(0);
    const auto scaled = [&](const float4 & v, float * sums) -> float {
        const float sum = pi_wave_sum(fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))));
        if (mine && lane == 0) sums[wave] = sum;
        __syncthreads();
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < NW; ++k) s += sums[k];
        return pi_inv_sqrt(s / (float)SIZE + p.eps);
    };
    const float f = p.mult * scaled(b, part[0]);
    x = make_float4(fmaf(f * b.x, w.x, x.x), fmaf(f * b.y, w.y, x.y), fmaf(f * b.z, w.z, x.z), fmaf(f * b.w, w.w, x.w));
    const float f2 = scaled(x, part[1]);
    if (mine) {
        *reinterpret_cast<float4 *>(p.x + base + col) = x;
        if (p.keep) *reinterpret_cast<float4 *>(p.keep + base + col) = x;
        const float v[4] = {f2 * x.x * next.x, f2 * x.y * next.y, f2 * x.z * next.z, f2 * x.w * next.w};
        store4((bf16 *)p.h + pi_ol_index(t, col), v, true, 4);
        store4(hs + col - c0, v, true, 4);
    }
    __syncthreads();
    float h[M][8];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const pi_u32x4 q = *reinterpret_cast<const pi_u32x4 *>(hs + m * 512 + lane * 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) { h[m][2 * e] = __uint_as_float(q[e] << 16); h[m][2 * e + 1] = __uint_as_float(q[e] & 0xFFFF0000u); }
    }
    float * sums = r.sums + (size_t)t * p.groups * r.E;
    for (int e0 = 0; e0 < r.E; e0 += kSrRows * kSrWaves) {
        if (e0) rows(e0);
        float s = 0.0f;                                             // lane k: the sum of row k
#pragma unroll
        for (int k = 0; k < kSrRows; ++k) {
            float d = 0.0f;
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    d = fmaf(__uint_as_float(ld[k][m][e] << 16), h[m][2 * e], d);
                    d = fmaf(__uint_as_float(ld[k][m][e] & 0xFFFF0000u), h[m][2 * e + 1], d);
                }
            d = pi_wave_sum(d);
            s = lane == k ? d : s;
        }
        const int e = e0 + wave + lane * kSrWaves;
        if (lane < kSrRows && e < r.E) __hip_atomic_store(sums + g * r.E + e, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // every wave waits for its own sums to have arrived before the workgroup says so: a barrier waits for LDS alone, and the release ahead of the count for the
    // stores of the wave that counts
    __builtin_amdgcn_s_waitcnt(0x0F70);                             // vmcnt(0)
    __syncthreads();
    if (tid == 0) last = __hip_atomic_fetch_add(r.arrived + t, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 == (unsigned int)p.groups;
    __syncthreads();
    if (!last) return;
    for (int e = tid; e < r.E; e += 64 * kSrWaves) {
        float s = 0.0f;
#pragma unroll 8
        for (int k = 0; k < p.groups; ++k) s += __hip_atomic_load(sums + k * r.E + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        z[e] = s;
    }
    if (tid == 0) __hip_atomic_store(r.arrived + t, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    RouteArgs a{z, r.E, r.top, 1, 1, nullptr, r.ids + (size_t)t * r.top, r.weights + (size_t)t * r.top};
    a.raw = true;
    route_token(a, 0, sm);
}

// An item of consecutive tokens of one run a workgroup: first the groups' scales of every row the item touches, then column by column the normed
// inputs of those rows and their convolution.
__host__ __device__ inline int conv_rows(int tokens, int taps) { return tokens + 2 * taps; }
template <typename ST>
__global__ __launch_bounds__(256) void conv_norm_kernel(pi_conv_norm p, int max_rows) {
    extern __shared__ __align__(16) float sm[];
    const int4 a = reinterpret_cast<const int4 *>(p.items)[2 * blockIdx.x], b = reinterpret_cast<const int4 *>(p.items)[2 * blockIdx.x + 1];
    const int t0 = a.x, n = a.y, off = a.z, len = a.w, slot = b.x, back = p.taps - 1, size = p.cols / p.groups;
    const bool head = off == 0, fresh = b.y != 0;
    const int before = min(off, back), run0 = t0 - off;
    // rows t0 - before .. t0 + n - 1, then (first item of a run) the run's last inputs behind them
    const int n_a = n + before, tail = head ? max(n, len - back) : len, rows = n_a + (head ? len - tail : 0);
    if (rows > max_rows) return;                       // (the launcher's bound)
    float * scale = sm, * part = sm + max_rows * p.groups;
    auto row = [&](int r) { return p.x + (size_t)(r < n_a ? t0 - before + r : run0 + tail + (r - n_a)) * p.cols; };
    group_scales(part, scale, rows, p.groups, p.cols, p.eps, row);
    float * state = p.state ? p.state + slot * p.slot_ld : nullptr;
    ST * h = (ST *)p.h;
    for (int c = threadIdx.x; c < p.cols; c += 256) {
        const int g = c / size;
        const float w = p.w[c], * tw = p.taps_w + c;
        auto input = [&](int i) -> float {             // the normed input at place i of the item (negative: before it)
            const int r = i + before;
            if (r >= 0) return p.x[(size_t)(t0 + i) * p.cols + c] * scale[r * p.groups + g] * w;
            const int s = off + i + back;              // before the run: row of the state
            return head && !fresh && s >= 0 ? state[(size_t)s * p.cols + c] : 0.0f;
        };
        for (int i = 0; i < n; ++i) {
            const float own = input(i);
            float v = 0.0f;
            for (int j = 0; j < back; ++j) v = fmaf(tw[(size_t)j * p.cols], input(i - back + j), v);
            v = fmaf(tw[(size_t)back * p.cols], own, v) + own;
            h[p.ol ? pi_ol_index(t0 + i, c) : (size_t)(t0 + i) * p.ld + c] = to_st<ST>(v);
        }
        if (!head || back == 0) continue;
        for (int s = 0; s < back; ++s) {               // ascending: an old row is read before it is overwritten
            const int i = len - back + s;              // place in the run
            float v;
            if (i < 0) v = fresh ? 0.0f : state[(size_t)(s + len) * p.cols + c];
            else if (i < n) v = input(i);
            else v = p.x[(size_t)(run0 + i) * p.cols + c] * scale[(n_a + i - tail) * p.groups + g] * w;
            state[(size_t)s * p.cols + c] = v;
        }
    }
}

// The same, four columns a thread, for up to BACK inputs ahead of a token and N >= BACK tokens of an item: a thread's inputs lie in registers, all requested together.
// groups: those of a workgroup, `size` columns each
template <typename ST, int BACK, int N>
__global__ __launch_bounds__(1024) void conv_norm_quads_kernel(pi_conv_norm p, int max_rows, int groups, int size) {
    extern __shared__ __align__(16) float sm[];
    const int4 a = reinterpret_cast<const int4 *>(p.items)[2 * blockIdx.x], b = reinterpret_cast<const int4 *>(p.items)[2 * blockIdx.x + 1];
    const int t0 = a.x, n = min(a.y, N), off = a.z, len = a.w, slot = b.x, lo = (int)blockIdx.y * groups * size, hi = lo + groups * size;
    const bool head = off == 0, fresh = b.y != 0;
    const int before = min(off, BACK), run0 = t0 - off, n_a = n + before, tail = head ? max(n, len - BACK) : len, rows = n_a + (head ? len - tail : 0);
    if (rows > max_rows) return;                       // (the launcher's bound)
    float * scale = sm, * part = sm + max_rows * groups;
    group_scales(part, scale, rows, groups, groups * size, p.eps, [&](int r) { return p.x + (size_t)(r < n_a ? t0 - before + r : run0 + tail + (r - n_a)) * p.cols + lo; });
    float * state = p.state ? p.state + slot * p.slot_ld : nullptr;
    ST * h = (ST *)p.h;
    for (int c = lo + threadIdx.x * 4; c < hi; c += blockDim.x * 4) {
        const int g = (c - lo) / size;
        const auto quad = [&](const float * q) { return *reinterpret_cast<const float4 *>(q + c); };
        float4 u[BACK + N], tw[BACK + 1];              // inputs: place k - BACK of the item
        const float4 w = quad(p.w);
#pragma unroll
        for (int j = 0; j <= BACK; ++j) tw[j] = quad(p.taps_w + (size_t)j * p.cols);
#pragma unroll
        for (int k = 0; k < BACK + N; ++k) {
            const int i = k - BACK;
            u[k] = make_float4(0, 0, 0, 0);
            if (i >= n) continue;
            if (i + before >= 0) u[k] = quad(p.x + (size_t)(t0 + i) * p.cols);
            else if (head && !fresh) u[k] = quad(state + (size_t)k * p.cols);
        }
#pragma unroll
        for (int k = 0; k < BACK + N; ++k) {
            const int r = k - BACK + before;
            if (r < 0 || r >= n_a) continue;
            const float f = scale[r * groups + g];
            u[k] = make_float4(u[k].x * f * w.x, u[k].y * f * w.y, u[k].z * f * w.z, u[k].w * f * w.w);
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (i >= n) break;
            float4 v = u[BACK + i];
#pragma unroll
            for (int j = 0; j <= BACK; ++j) {
                const float4 q = u[i + j];
                v = make_float4(fmaf(tw[j].x, q.x, v.x), fmaf(tw[j].y, q.y, v.y), fmaf(tw[j].z, q.z, v.z), fmaf(tw[j].w, q.w, v.w));
            }
            const float o[4] = {v.x, v.y, v.z, v.w};
            store4(h + (p.ol ? pi_ol_index(t0 + i, c) : (size_t)(t0 + i) * p.ld + c), o, true, 4);
        }
        if (!head || BACK == 0) continue;
#pragma unroll
        for (int s = 0; s < BACK; ++s) {
            const int i = len - BACK + s;              // place in the run
            float4 v = make_float4(0, 0, 0, 0);
            if (i >= n) {
                const float f = scale[(n_a + i - tail) * groups + g];
                const float4 q = quad(p.x + (size_t)(run0 + i) * p.cols);
                v = make_float4(q.x * f * w.x, q.y * f * w.y, q.z * f * w.z, q.w * f * w.w);
            } else {
#pragma unroll
                for (int k = 0; k < BACK + N; ++k) if (k == BACK + i) v = u[k];
            }
            *reinterpret_cast<float4 *>(state + (size_t)s * p.cols + c) = v;
        }
    }
}
// The sum that closes a layer (sum_norm_quads_kernel's) and the next layer's norm and convolution in one launch, for items that are whole runs: nothing of a
// run's group is needed elsewhere.  A token after the other, a group a workgroup, the run's inputs in registers.  Bound by latency like both: 4096 columns, one token
// 4.4 + 4.9 -> 4.7 us.
template <typename ST, int BACK>
__global__ __launch_bounds__(1024) void sum_conv_kernel(pi_sum_norm p, pi_conv_norm c) {
    __shared__ float part[2][16];
    const int4 a = reinterpret_cast<const int4 *>(c.items)[2 * blockIdx.x], b = reinterpret_cast<const int4 *>(c.items)[2 * blockIdx.x + 1];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6, size = p.cols / p.groups, col = (int)blockIdx.y * size + (int)threadIdx.x * 4;
    const auto quad = [&](const float * v) { return *reinterpret_cast<const float4 *>(v + col); };
    const float4 w_after = quad(p.w), w = quad(c.w);
    float4 tw[BACK + 1], past[BACK + 1];                            // (the last of past is the token's own)
#pragma unroll
    for (int j = 0; j <= BACK; ++j) tw[j] = quad(c.taps_w + (size_t)j * p.cols);
    float * state = c.state ? c.state + b.x * c.slot_ld : nullptr;
#pragma unroll
    for (int j = 0; j < BACK; ++j) past[j] = b.y ? make_float4(0, 0, 0, 0) : quad(state + (size_t)j * p.cols);
    const auto scaled = [&](const float4 & v, float * sums) -> float {
        const float sum = pi_wave_sum(fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))));
        if (lane == 0) sums[wave] = sum;
        __syncthreads();
        float s = 0.0f;
        for (int k = 0; k < waves; ++k) s += sums[k];
        return pi_inv_sqrt(s / (float)size + p.eps);
    };
    for (int i = 0; i < a.y; ++i) {
        const size_t base = (size_t)(a.x + i) * p.cols;
        const float4 m = quad(p.mix + base);
        float4 x = quad(p.x + base);
        const float f = p.mult * scaled(m, part[0]);
        x = make_float4(fmaf(f * m.x, w_after.x, x.x), fmaf(f * m.y, w_after.y, x.y), fmaf(f * m.z, w_after.z, x.z), fmaf(f * m.w, w_after.w, x.w));
        *reinterpret_cast<float4 *>(p.x + base + col) = x;
        if (p.keep) *reinterpret_cast<float4 *>(p.keep + base + col) = x;
        const float g = scaled(x, part[1]);                         // (part[0] has been read by all behind this barrier)
        past[BACK] = make_float4(x.x * g * w.x, x.y * g * w.y, x.z * g * w.z, x.w * g * w.w);
        float4 v = past[BACK];
#pragma unroll
        for (int j = 0; j <= BACK; ++j) v = make_float4(fmaf(tw[j].x, past[j].x, v.x), fmaf(tw[j].y, past[j].y, v.y), fmaf(tw[j].z, past[j].z, v.z), fmaf(tw[j].w, past[j].w, v.w));
        const float o[4] = {v.x, v.y, v.z, v.w};
        store4((ST *)c.h + (c.ol ? pi_ol_index(a.x + i, col) : (size_t)(a.x + i) * c.ld + col), o, true, 4);
#pragma unroll
        for (int j = 0; j < BACK; ++j) past[j] = past[j + 1];
    }
#pragma unroll
    for (int j = 0; j < BACK; ++j) *reinterpret_cast<float4 *>(state + (size_t)j * p.cols + col) = past[j];
}
template <typename ST> void launch_sum_conv(const pi_sum_norm & p, const pi_conv_norm & c, hipStream_t st) {
    const dim3 grid(c.n_items, p.groups), block(p.cols / p.groups / 4);
    switch (c.taps) {
        case 1: hipLaunchKernelGGL((sum_conv_kernel<ST, 0>), grid, block, 0, st, p, c); break;
        case 2: hipLaunchKernelGGL((sum_conv_kernel<ST, 1>), grid, block, 0, st, p, c); break;
        case 3: hipLaunchKernelGGL((sum_conv_kernel<ST, 2>), grid, block, 0, st, p, c); break;
        case 4: hipLaunchKernelGGL((sum_conv_kernel<ST, 3>), grid, block, 0, st, p, c); break;
        default: hipLaunchKernelGGL((sum_conv_kernel<ST, 4>), grid, block, 0, st, p, c);
    }
}
template <typename ST> bool launch_conv_quads(const pi_conv_norm & p, int rows, size_t lds, hipStream_t st) {
    if ((p.cols / p.groups) % 4 || p.ld % 4 || p.slot_ld % 4 || p.taps > 5) return false;
    // As many workgroups of whole groups as run at once: two a unit, one of 1024 threads (whose registers leave no room for another: 700 tokens of 6144 columns in 4 groups, 350
    // workgroups of two groups 14.5 us, 175 of all 11.8).  One token's 160 KB are 6.6 us for one unit, 4.7 for eight.
    const int size = p.cols / p.groups;
    const auto threads = [&](int groups) { return groups * size > 2048 ? 1024 : groups * size > 1024 ? 512 : 256; };
    int groups = p.groups;
    for (int d = 2; d <= p.groups && p.n_items * d <= 2 * pi::compute_units(); ++d)
        if (p.groups % d == 0 && p.n_items * d <= pi::compute_units() * (threads(p.groups / d) > 512 ? 1 : 2)) groups = p.groups / d;
    const dim3 grid(p.n_items, p.groups / groups), block(threads(groups));
    switch (p.taps) {
        case 1: hipLaunchKernelGGL((conv_norm_quads_kernel<ST, 0, 4>), grid, block, lds, st, p, rows, groups, size); break;
        case 2: hipLaunchKernelGGL((conv_norm_quads_kernel<ST, 1, 4>), grid, block, lds, st, p, rows, groups, size); break;
        case 3: hipLaunchKernelGGL((conv_norm_quads_kernel<ST, 2, 4>), grid, block, lds, st, p, rows, groups, size); break;
        case 4: hipLaunchKernelGGL((conv_norm_quads_kernel<ST, 3, 4>), grid, block, lds, st, p, rows, groups, size); break;
        default: hipLaunchKernelGGL((conv_norm_quads_kernel<ST, 4, 4>), grid, block, lds, st, p, rows, groups, size);
    }
    return true;
}

}  // namespace

extern "C" {

int pi_k_sum_norm(int type, const pi_sum_norm * p, pi_stream_t stream) {
    if (!p || !p->x || p->T <= 0 || p->cols <= 0 || p->groups <= 0 || p->cols % p->groups || (p->w && (p->rows || !p->mix == !p->y || (p->y && (!p->inv || p->top <= 0)))) || (!p->w && !p->h) ||
        (p->h && (!p->w_next || p->ld < p->cols)))
        return pi::fail(PI_E_ARG, "pi_k_sum_norm: bad arguments");
    if (p->cols > kNormMaxCols || p->groups > 1024) return pi::fail(PI_E_UNSUPPORTED, "pi_k_sum_norm: up to 32768 columns in up to 1024 groups");
    if (p->h && p->ol && (type != PI_TYPE_BF16 || p->T > kBtMaxT || p->ld % 8)) return pi::fail(PI_E_ARG, "pi_k_sum_norm: operand layout needs BF16, T <= 16, ld % 8 == 0");
    if (type == PI_TYPE_BF16 ? launch_sum_quads<bf16>(*p, (hipStream_t)stream) : type == PI_TYPE_F32 && launch_sum_quads<float>(*p, (hipStream_t)stream)) return pi::check_launch("pi_k_sum_norm");
    const int block = p->cols > 2048 ? 1024 : p->cols > 1024 ? 512 : 256;
    const size_t lds = sizeof(float) * ((size_t)(p->cols + 3) / 4 * 4 + p->groups + group_parts(1, p->groups, block / 64));
    static bool raised = false;
    if (!raised) {
        PI_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&sum_norm_kernel<bf16>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
        PI_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&sum_norm_kernel<float>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
        raised = true;
    }
    if (type == PI_TYPE_BF16) hipLaunchKernelGGL(sum_norm_kernel<bf16>, dim3(p->T), dim3(block), lds, (hipStream_t)stream, *p);
    else if (type == PI_TYPE_F32) hipLaunchKernelGGL(sum_norm_kernel<float>, dim3(p->T), dim3(block), lds, (hipStream_t)stream, *p);
    else return pi::fail(PI_E_UNSUPPORTED, "pi_k_sum_norm: type");
    return pi::check_launch("pi_k_sum_norm");
}

int pi_k_sum_norm_route_supported(int T, int cols, int groups, int n_expert) {
    return T > 0 && T <= kBtMaxT && groups > 0 && groups <= kSrGroups && n_expert > 0 && n_expert <= kSrExperts && (cols == 512 * groups || cols == 1024 * groups) && n_expert * (cols / groups) <= 65536;
}

int pi_k_sum_norm_route(const pi_sum_norm * p, const void * router, int ld_router, int n_expert, int n_top, int32_t * ids, float * weights, float * sums, uint32_t * arrived, pi_stream_t stream) {
    if (!p || !p->x || !p->mix || !p->w || !p->w_next || !p->h || p->rows || p->y || !p->ol || p->ld < p->cols || p->ld % 8 || !router || ld_router < p->cols || ld_router % 8 || n_top <= 0 ||
        n_top > n_expert || !ids || !weights || !sums || !arrived)
        return pi::fail(PI_E_ARG, "pi_k_sum_norm_route: bad arguments");
    if (!pi_k_sum_norm_route_supported(p->T, p->cols, p->groups, n_expert)) return pi::fail(PI_E_UNSUPPORTED, "pi_k_sum_norm_route: groups of 512 or 1024 columns, up to 65536 values of the router a group");
    const SumRoute r{(const bf16 *)router, ld_router, n_expert, n_top, ids, weights, sums, arrived};
    if (p->cols == 512 * p->groups) hipLaunchKernelGGL(sum_norm_route_kernel<1>, dim3(p->T, p->groups), dim3(64 * kSrWaves), 0, (hipStream_t)stream, *p, r);
    else hipLaunchKernelGGL(sum_norm_route_kernel<2>, dim3(p->T, p->groups), dim3(64 * kSrWaves), 0, (hipStream_t)stream, *p, r);
    return pi::check_launch("pi_k_sum_norm_route");
}

int pi_k_conv_tokens(int T, int taps) { return T <= 16 ? (taps > 2 ? taps - 1 : 1) : taps > 5 ? taps - 1 : 4; }

int pi_k_conv_norm(int type, const pi_conv_norm * p, pi_stream_t stream) {
    if (!p || !p->x || !p->w || !p->taps_w || !p->items || !p->h || p->T <= 0 || p->n_items <= 0 || p->cols <= 0 || p->groups <= 0 || p->cols % p->groups || p->taps <= 0 || p->ld < p->cols ||
        (p->taps > 1 && (!p->state || p->slot_ld < (size_t)(p->taps - 1) * p->cols)))
        return pi::fail(PI_E_ARG, "pi_k_conv_norm: bad arguments");
    if (p->ol && (type != PI_TYPE_BF16 || p->T > kBtMaxT || p->ld % 8)) return pi::fail(PI_E_ARG, "pi_k_conv_norm: operand layout needs BF16, T <= 16, ld % 8 == 0");
    const int rows = conv_rows(pi_k_conv_tokens(p->T, p->taps), p->taps);
    const size_t lds = sizeof(float) * ((size_t)rows * p->groups + group_parts(rows, p->groups, 16) + 16);
    if (lds > 64 * 1024) return pi::fail(PI_E_UNSUPPORTED, "pi_k_conv_norm: taps x groups");
    if (type != PI_TYPE_BF16 && type != PI_TYPE_F32) return pi::fail(PI_E_UNSUPPORTED, "pi_k_conv_norm: type");
    hipStream_t st = (hipStream_t)stream;
    if (type == PI_TYPE_BF16 ? launch_conv_quads<bf16>(*p, rows, lds, st) : launch_conv_quads<float>(*p, rows, lds, st)) return pi::check_launch("pi_k_conv_norm");
    if (type == PI_TYPE_BF16) hipLaunchKernelGGL(conv_norm_kernel<bf16>, dim3(p->n_items), dim3(256), lds, st, *p, rows);
    else hipLaunchKernelGGL(conv_norm_kernel<float>, dim3(p->n_items), dim3(256), lds, st, *p, rows);
    return pi::check_launch("pi_k_conv_norm");
}

int pi_k_sum_conv_supported(int cols, int groups, int taps, int ld, size_t slot_ld) {
    return cols > 0 && groups > 0 && cols % groups == 0 && cols / groups % 256 == 0 && cols / groups <= 4096 && taps > 0 && taps <= 5 && ld >= cols && ld % 4 == 0 && slot_ld % 4 == 0;
}

int pi_k_sum_conv(int type, const pi_sum_norm * p, const pi_conv_norm * c, pi_stream_t stream) {
    if (!p || !c || !p->x || !p->mix || !p->w || p->y || p->rows || p->h || p->T <= 0 || !c->w || !c->taps_w || !c->items || !c->h || c->n_items <= 0 || c->x != p->x || c->T != p->T ||
        c->cols != p->cols || c->groups != p->groups || c->eps != p->eps || (c->taps > 1 && (!c->state || c->slot_ld < (size_t)(c->taps - 1) * c->cols)))
        return pi::fail(PI_E_ARG, "pi_k_sum_conv: bad arguments");
    if (c->ol && (type != PI_TYPE_BF16 || p->T > kBtMaxT || c->ld % 8)) return pi::fail(PI_E_ARG, "pi_k_sum_conv: operand layout needs BF16, T <= 16, ld % 8 == 0");
    if (!pi_k_sum_conv_supported(p->cols, p->groups, c->taps, c->ld, c->slot_ld) || (type != PI_TYPE_BF16 && type != PI_TYPE_F32))
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_sum_conv: groups of whole 256 columns, up to 4096, up to five taps");
    if (type == PI_TYPE_BF16) launch_sum_conv<bf16>(*p, *c, (hipStream_t)stream);
    else launch_sum_conv<float>(*p, *c, (hipStream_t)stream);
    return pi::check_launch("pi_k_sum_conv");
}

}  // extern "C"
