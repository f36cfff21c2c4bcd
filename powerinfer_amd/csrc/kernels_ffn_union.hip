// The sparse FFN of a long prompt chunk over the neurons that fire for one of its tokens: predictor bits, their list, gate and up of the listed neurons, and the
// down projection that goes through the list again.  11008 neurons, 4096 columns, 2047 tokens, us: bits 50, list 5, gate and up of all neurons 303 (1.22 PFLOP/s)
// and of half of them 160, down projection 160 (the library's product over all of them 170) and 92.  What bounds the products is what the tiles bring to
// LDS: without these copies 303 us are about 245.
#include "ffn_wide.hpp"
#include "runtime.hpp"
#include "../../include/powerinfer_hip.h"

#include <algorithm>

namespace {

constexpr int kUnionMost = 32768;            // neurons: a thread of the list's workgroups has 32
constexpr int kUnionLeast = 256;             // listed ones at least (four stages of the down projection's columns)

// The neurons that fire for a token of the chunk in ascending order, filled up to a multiple of 128 with one of them (h is 0 there), and the predictor's bits in that
// order.  A workgroup for 16 tokens' bits, one for the list; each finds the neurons' places by itself.  n_active: of the last token.
// Bound by latency (a few KB a workgroup): 4 us, 10 for 2047 tokens of 11008 neurons in one that went through a tile's words bit by bit.
// told (its word may be null): gets their number, 16 bits.  From `all_from` neurons on the list is all of them, and nobody packs anything (bits one by one for every neuron: 26 us for 32768 of them).
__global__ __launch_bounds__(1024) void ffn_union_list_kernel(const uint32_t * __restrict__ any, int any_rows, const unsigned long long * __restrict__ mask, int T, int ff, int all_from, pi::HostAsk told, int32_t * __restrict__ list,
                                                              int32_t * __restrict__ count, unsigned long long * __restrict__ packed, int32_t * __restrict__ n_active) {
    extern __shared__ __align__(16) uint16_t bits[];                    // of the listed neurons, as a tile's words hold them
    __shared__ int sums[16], last;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, words = ff / 32, tile = blockIdx.x;
    ulonglong2 w[4] = {};
    uint32_t fires = 0;
    if (t < words) {
        const ulonglong2 * in = reinterpret_cast<const ulonglong2 *>(mask + (size_t)min(tile, (T - 1) / 16) * (ff / 4) + 8 * t);
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = in[k];
#pragma unroll 8
        for (int r = 0; r < any_rows; ++r) fires |= any[(size_t)r * words + t];
    }
    if (t == 0) last = 0;                                               // (nobody fires)
    int at = __popc(fires);
    const int own = at;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(at, o, 64); if (lane >= o) at += v; }
    if (lane == 63) sums[wave] = at;
    __syncthreads();
    int n = 0;
    for (int k = 0; k < 16; ++k) { if (k == wave) at += n; n += sums[k]; }
    at -= own;
    const int padded = n >= all_from ? ff : max(kUnionLeast, (n + 127) / 128 * 128);
    const auto place = [](int p) { return ((p >> 4) * 4 + (p & 3)) * 4 + (p >> 2 & 3); };
    if (padded < ff && n + t < padded) bits[place(n + t)] = 0;
    if (own && at + own == n) last = 32 * t + 31 - __clz(fires);
    const unsigned long long word[8] = {w[0].x, w[0].y, w[1].x, w[1].y, w[2].x, w[2].y, w[3].x, w[3].y};
    if (tile == (int)gridDim.x - 1) {                                   // the list
        if (padded == ff) {
            for (int p = t; p < ff; p += 1024) list[p] = p;
            if (t == 0) { *count = ff; if (told.word) __hip_atomic_store(told.word, told.tag | (uint32_t)ff, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
            return;
        }
        for (int p = at; fires; fires &= fires - 1) list[p++] = 32 * t + __builtin_ctz(fires);
        __syncthreads();
        if (n + t < padded) list[n + t] = last;
        if (t == 0) { *count = padded; if (told.word) __hip_atomic_store(told.word, told.tag | (uint32_t)padded, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
        return;
    }
    if (padded < ff)
#pragma unroll
        for (int b = 0, p = at; b < 32; ++b)
            if (fires >> b & 1) bits[place(p++)] = (uint16_t)(word[(b >> 4) * 4 + (b & 3)] >> 16 * (b >> 2 & 3));
    if (n_active && tile == (T - 1) / 16) {                             // (count_active_kernel has the same word)
        int mine = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) mine += __popcll(word[k] & 0x0001000100010001ull << ((T - 1) & 15));
        mine = (int)pi_wave_sum((float)mine);
        __syncthreads();
        if (lane == 0) sums[wave] = mine;
        __syncthreads();
        if (t == 0) { int all = 0; for (int k = 0; k < 16; ++k) all += sums[k]; *n_active = all; }
    }
    if (padded == ff) return;
    __syncthreads();
    for (int k = t; k < padded / 8; k += 1024) reinterpret_cast<uint4 *>(packed + (size_t)tile * (padded / 4))[k] = reinterpret_cast<const uint4 *>(bits)[k];
}

// How many may stay silent for all of them to be gone through as they lie, as ffn_wide_kernel does: what the list costs (its packing, and rows looked up one by one) is 15 to 50 us, what it
// saves goes with the tokens.  Four layers, us, list / all.  All neurons fire: 7B 400 tokens 1194 / 1172, 13B 140 1200 / 1185, 300 1531 / 1463, 1800 4623 / 4574, 40B 57 1628 / 1520, 600 3705 /
// 3617, 1900 8491 / 8367.  0.95 of them: 13B 90 tokens 1088 / 1101, 300 1508 / 1466, 40B 18 1547 / 1483, 320 2567 / 2479; but 13B 1800 4476 / 4537, 40B 1900 8294 / 8427.
inline int union_silent(int ff, int T) { return ff / (T > 512 ? 32 : 16); }

// gate, up and h of the listed neurons: h [T][count]
template <bool PAIRS> __global__ __launch_bounds__(512, 1) void ffn_wide_union_kernel(FfnProduct<PAIRS, true, true> prod, const unsigned long long * __restrict__ mask, const int32_t * __restrict__ count) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = *count;
    const WideDeal deal(PAIRS ? 2 * n : n, (prod.T + kGwN - 1) / kGwN, kGwBand);
    if (n == prod.ff) {
        gemm_wide<__half>(FfnProduct<PAIRS, true, false>{prod.up, prod.gate, prod.x, nullptr, prod.thr, prod.h16, n, prod.cols, prod.T, prod.nk, mask, nullptr}, deal, smem);
        return;
    }
    prod.ff = n;
    gemm_wide<__half>(prod, deal, smem);
}

// How the down projection's workgroups share its units (256 rows of a token tile): each XCD a contiguous range, band by band, as WideDeal has it.  What does not fill
// the XCD's workgroups once more is shared by up to eight of them a unit: up to four have a part of its neurons each and leave 32-bit sums in parts,
// which are added behind them in their order, or (and) two have half of its rows each.  4096 columns, 5504 listed neurons, us, halves only / parts: 64 tokens 53 / 25, 200 56 / 29,
// 400 57 / 39, 700 61 / 53; 5120 columns of 13824, 1800 tokens 299 / 242; 8192 of 14208, 300 tokens 142 / 101.
constexpr int kUnionParts = 4;
struct DownDeal {
    int n_tiles, nx, per, rounds, rest, parts, halves, count, xcd, slot, slots;
    __host__ __device__ __forceinline__ DownDeal(int rows, int n_tiles_, bool room, int xcd_, int slot_, int slots_) {
        n_tiles = n_tiles_; nx = rows / kGwM; xcd = xcd_; slot = slot_; slots = slots_;
        per = (n_tiles * nx + 7) / 8;
        const int left = n_tiles * nx - xcd * per, n = left < 0 ? 0 : left < per ? left : per, share = n % slots ? slots / (n % slots) : 0;
        rounds = n / slots; rest = n % slots;
        halves = share >= 2 * kUnionParts || (share >= 2 && !room) ? 2 : 1;
        parts = !room || share < 2 ? 1 : share < kUnionParts ? share : kUnionParts;
        count = rounds + (slot < rest * parts * halves ? 1 : 0);
    }
    // the place of the XCD's u-th unit
    __host__ __device__ __forceinline__ void tile(int u, int & ty, int & row0) const {
        const int at = xcd * per + u, b0 = at / (kGwBand * nx) * kGwBand, high = n_tiles - b0 < kGwBand ? n_tiles - b0 : kGwBand, in = at - b0 * nx;
        ty = b0 + in % high; row0 = in / high * kGwM;
    }
    // the workgroup's c-th: and which part of its neurons (of `parts`, 1: all)
    __host__ __device__ __forceinline__ void unit(int c, int & ty, int & row0, int & rows, int & part, int & of) const {
        const bool last = c >= rounds;
        const int sub = slot % (parts * halves);
        tile(last ? rounds * slots + slot / (parts * halves) : c * slots + slot, ty, row0);
        rows = last && halves == 2 ? kGwM / 2 : kGwM;
        part = last ? sub % parts : 0; of = last ? parts : 1;
        if (last) row0 += sub / parts * (kGwM / 2);
    }
};

// DownDeal, and where what does not fill the XCD's workgroups once more is from a half to three quarters of them: its units in three or four parts, which the workgroups take in two
// or three turns, all units' first parts first (workgroups side by side go through the same rows; an equal range of stages for each, wherever it begins, is slower than leaving the
// others idle: 40B, 600 tokens, four layers 3600 -> 4000 us).  Prompts of four layers, us, whole / in turns, all neurons firing: 13B 800 tokens 2597 / 2469, 1000 2948 / 2780, 40B 520 3521 / 3312, 600
// 3710 / 3455, 1600 7813 / 7534; half of them: 13B 800 2028 / 2002, 40B 600 2765 / 2639.  Shorter lists gain less than the sums take (7B, 86 stages of 172, 1200 tokens: 1749 / 1760).  The launch that adds the parts comes whether this list is long enough or not, so it is asked for by the longest one.
constexpr int kUnionMostStages = 64, kUnionStages = 24;               // of a part: of the longest list, and of this one
struct DownSplit {
    DownDeal deal;
    int parts, count;
    bool turns;
    // most: stages of all neurons (no room for parts: 0), nk: of the listed ones
    __host__ __device__ __forceinline__ DownSplit(const DownDeal & d, int most, int nk) : deal(d) {
        parts = d.rest * 3 <= d.slots * 2 ? 3 : 4;
        turns = d.rest * 2 > d.slots && d.rest * 4 <= d.slots * 3 && most >= kUnionMostStages * parts && nk >= kUnionStages * parts;
        if (!turns) parts = d.parts;
        count = turns ? d.rounds + (d.rest * parts - d.slot + d.slots - 1) / d.slots : d.count;
    }
    __host__ __device__ __forceinline__ void unit(int c, int & ty, int & row0, int & rows, int & part, int & of) const {
        if (!turns || c < deal.rounds) return deal.unit(c, ty, row0, rows, part, of);
        const int at = deal.slot + (c - deal.rounds) * deal.slots;
        deal.tile(deal.rounds * deal.slots + at % deal.rest, ty, row0);
        rows = kGwM; part = at / deal.rest; of = parts;
    }
};

// out[t][c] = sum over the listed neurons of h[t][k] down_t[list[k]][c], and what is added to it
struct DownProduct {
    static constexpr bool kPairs = false, kList = false, kTurned = true;
    static constexpr int kM = kGwM, kN = kGwN;
    const __half * down, * h; const int32_t * turned; const float * add1, * add2; float * out;
    int rows, T; uint32_t col_bytes; int most; float * parts[kUnionParts - 1];
    int n, nk;                                                          // listed neurons, stages of them
    __device__ __forceinline__ bool read_once(const WidePlace &) const { return false; }
    __device__ __forceinline__ int first(const WidePlace & p) const { return nk * (p.grp & 7) / (p.grp >> 3); }
    __device__ __forceinline__ int stages(const WidePlace & p) const { return nk * ((p.grp & 7) + 1) / (p.grp >> 3) - first(p); }
    __device__ __forceinline__ WidePlace place(const DownSplit & deal, int c) const {      // (grp: which part, and of how many)
        WidePlace p;
        int ty, part, of;
        deal.unit(c, ty, p.row0, p.rows, part, of);
        p.grp = part | of << 3; p.lo = ty * kGwN; p.n = min(T - p.lo, kGwN);
        return p;
    }
    __device__ __forceinline__ const unsigned char * base_a(const WidePlace & p, int) const { return (const unsigned char *)(down + p.row0); }
    __device__ __forceinline__ const unsigned char * base_b(const WidePlace & p) const { return (const unsigned char *)(h + (size_t)p.lo * n); }
    __device__ __forceinline__ size_t off_b(const WidePlace &, int r) const { return (size_t)r * n * 2; }
    template <int MT> __device__ __forceinline__ void store(const WidePlace & p, int rb, int tb, const pi_f4 (&acc)[MT][4], unsigned char *, int lane) const {
        asm volatile("" : "+v"(lane));                 // what follows is computed here, not kept in registers across the products
        const int i = lane & 15, q = lane >> 4;
        const auto at = [&](int nn) { return (size_t)(p.lo + min(tb + nn * 16 + i, p.n - 1)) * rows + p.row0 + rb + 4 * q; };
        if (p.grp >> 3 > 1) {
            const int part = p.grp & 7;
            float * to = part == 0 ? out : part == 1 ? parts[0] : part == 2 ? parts[1] : parts[2];
#pragma unroll
            for (int nn = 0; nn < 4; ++nn) {
                if (tb + nn * 16 + i >= p.n) continue;
#pragma unroll
                for (int m = 0; m < MT; ++m) *reinterpret_cast<pi_f4 *>(to + at(nn) + m * 16) = acc[m][nn];
            }
            return;
        }
        float4 v[2][MT];                               // a token's are requested under the sums of the one before
        const auto fetch = [&](int nn) {
#pragma unroll
            for (int m = 0; m < MT; ++m) v[nn & 1][m] = *reinterpret_cast<const float4 *>(add1 + at(nn) + m * 16);
        };
        fetch(0);
#pragma unroll
        for (int nn = 0; nn < 4; ++nn) {
            if (nn < 3) fetch(nn + 1);
            const bool mine = tb + nn * 16 + i < p.n;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float4 a = v[nn & 1][m];
                float4 y = make_float4(__fadd_rn(acc[m][nn][0], a.x), __fadd_rn(acc[m][nn][1], a.y), __fadd_rn(acc[m][nn][2], a.z), __fadd_rn(acc[m][nn][3], a.w));
                if (add2) {
                    const float4 o = *reinterpret_cast<const float4 *>(add2 + at(nn) + m * 16);
                    y = make_float4(__fadd_rn(y.x, o.x), __fadd_rn(y.y, o.y), __fadd_rn(y.z, o.z), __fadd_rn(y.w, o.w));
                }
                if (mine) *reinterpret_cast<float4 *>(out + at(nn) + m * 16) = y;
            }
        }
    }
};
__global__ __launch_bounds__(512, 1) void ffn_union_down_kernel(DownProduct a, const int32_t * __restrict__ count) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = *count;
    const DownDeal deal(a.rows, (a.T + kGwN - 1) / kGwN, a.most > 0, (int)blockIdx.x % 8, (int)blockIdx.x / 8, (int)gridDim.x / 8);
    const DownProduct prod{a.down, a.h, a.turned, a.add1, a.add2, a.out, a.rows, a.T, a.col_bytes, a.most, {a.parts[0], a.parts[1], a.parts[2]}, n, n / kGtBK};
    gemm_wide<__half>(prod, DownSplit(deal, a.most, prod.nk), smem);
}
// (count: null where no list has turns)  Units that were shared: out += the other parts in their order, and what is added to them; 1024 values of a unit a workgroup, four a thread
constexpr int kUnionGrid = 256;              // workgroups of the down projection
__global__ __launch_bounds__(256) void ffn_union_sum_kernel(DownProduct a, const int32_t * __restrict__ count) {
    const DownDeal deal(a.rows, (a.T + kGwN - 1) / kGwN, a.most > 0, (int)blockIdx.z, 0, kUnionGrid / 8);
    const int parts = count ? DownSplit(deal, a.most, *count / kGtBK).parts : deal.parts;
    if (parts == 1 || (int)blockIdx.y >= deal.rest) return;
    int ty, row0;
    deal.tile(deal.rounds * deal.slots + (int)blockIdx.y, ty, row0);
    const int t = ty * kGwN + (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6);
    if (t >= a.T) return;
    const size_t o = (size_t)t * a.rows + row0 + (threadIdx.x & 63) * 4;
    float4 v = *reinterpret_cast<const float4 *>(a.out + o), b[kUnionParts - 1] = {}, a1 = *reinterpret_cast<const float4 *>(a.add1 + o), a2{};
#pragma unroll
    for (int k = 0; k < kUnionParts - 1; ++k)
        if (k + 1 < parts) b[k] = *reinterpret_cast<const float4 *>(a.parts[k] + o);
    if (a.add2) a2 = *reinterpret_cast<const float4 *>(a.add2 + o);
#pragma unroll
    for (int k = 0; k < kUnionParts - 1; ++k)
        if (k + 1 < parts) { v.x += b[k].x; v.y += b[k].y; v.z += b[k].z; v.w += b[k].w; }
    v = make_float4(__fadd_rn(v.x, a1.x), __fadd_rn(v.y, a1.y), __fadd_rn(v.z, a1.z), __fadd_rn(v.w, a1.w));
    if (a.add2) v = make_float4(__fadd_rn(v.x, a2.x), __fadd_rn(v.y, a2.y), __fadd_rn(v.z, a2.z), __fadd_rn(v.w, a2.w));
    *reinterpret_cast<float4 *>(a.out + o) = v;
}

template <typename K> int raise_lds(K kernel, int bytes) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    return e == hipSuccess ? PI_OK : pi::hip_fail(e, "pi_k_ffn_union_f16: LDS size");
}
size_t up16(size_t n) { return (n + 15) / 16 * 16; }
// where things lie in the caller's scratch
struct UnionScratch {
    size_t packed, any, list, count, bytes;
    UnionScratch(int ff, int T) {
        const size_t mask = (size_t)((T + 15) / 16) * ff * 2;
        packed = mask; any = packed + mask; list = any + up16((size_t)((T + 63) / 64) * (ff / 8)); count = list + (size_t)ff * 4; bytes = count + 16;
    }
};
int wide_tiles(int rows, int T) { return (rows + kGwM - 1) / kGwM * ((T + kGwN - 1) / kGwN); }

}  // namespace

extern "C" {

int pi_k_ffn_union_supported(int ff, int rank, int cols) {
    return ff >= kUnionLeast && ff % 128 == 0 && ff <= kUnionMost && cols % 256 == 0 && pi_k_ffn_wide_supported(ff, cols) && pi_k_ffn_wide_supported(ff, rank);
}
size_t pi_k_ffn_union_scratch(int ff, int T) { return UnionScratch(ff, T).bytes; }

}  // extern "C"
namespace pi {
int ffn_union_hidden(const void * fc2_f16, int rank, const void * hid_f16, const void * up_f16, const void * gate_f16, int ff, int cols, const void * xn_f16, int T, float threshold, void * scratch,
                     void * h_f16, int32_t * n_active, const HostAsk & told, pi_stream_t stream) {
    if (!fc2_f16 || !hid_f16 || !up_f16 || !xn_f16 || !scratch || !h_f16 || T <= 0) return fail(PI_E_ARG, "pi_k_ffn_union_f16: bad arguments");
    if (!pi_k_ffn_union_supported(ff, rank, cols)) return fail(PI_E_UNSUPPORTED, "pi_k_ffn_union_f16: ff a multiple of 128 from 256 to 32768, cols one of 256, rank one of 64 from 256 on");
    if ((((uintptr_t)fc2_f16 | (uintptr_t)hid_f16 | (uintptr_t)up_f16 | (uintptr_t)gate_f16 | (uintptr_t)xn_f16 | (uintptr_t)scratch | (uintptr_t)h_f16) & 15) != 0)
        return fail(PI_E_ARG, "pi_k_ffn_union_f16: operands must be 16-byte aligned");
    const long long units = (long long)((2 * (long long)ff + kGwM - 1) / kGwM) * ((T + kGwN - 1) / kGwN);
    if (units > (1 << 30)) return fail(PI_E_ARG, "pi_k_ffn_union_f16: too many tiles");
    static const int raised = [] {
        int rc = raise_lds(ffn_union_list_kernel, 2 * kUnionMost);
        if (rc == PI_OK) rc = raise_lds(ffn_wide_union_kernel<true>, kGwLds);
        return rc == PI_OK ? raise_lds(ffn_wide_union_kernel<false>, kGwLds) : rc;
    }();
    if (raised != PI_OK) return raised;
    const UnionScratch at(ff, T);
    unsigned char * s = (unsigned char *)scratch;
    unsigned long long * mask = (unsigned long long *)s, * packed = (unsigned long long *)(s + at.packed);
    int32_t * list = (int32_t *)(s + at.list), * count = (int32_t *)(s + at.count);
    hipStream_t st = (hipStream_t)stream;
    if (const int rc = predictor_bits(fc2_f16, ff, rank, hid_f16, T, threshold, mask, s + at.any, stream)) return rc;
    hipLaunchKernelGGL(ffn_union_list_kernel, dim3((T + 15) / 16 + 1), dim3(1024), (size_t)ff * 2, st, (const uint32_t *)(s + at.any), (T + 63) / 64, mask, T, ff, ff - union_silent(ff, T), told, list, count, packed,
                       n_active);
    const auto wide = [&](auto pairs) {
        constexpr bool P = decltype(pairs)::value;
        hipLaunchKernelGGL(ffn_wide_union_kernel<P>, dim3(wide_blocks(wide_tiles(P ? 2 * ff : ff, T))), dim3(512), kGwLds, st,
                           FfnProduct<P, true, true>{(const __half *)up_f16, (const __half *)gate_f16, (const __half *)xn_f16, nullptr, threshold, (__half *)h_f16, ff, cols, T, cols / kGtBK, packed, list}, mask, count);
    };
    if (gate_f16) wide(std::true_type{}); else wide(std::false_type{});
    return check_launch("pi_k_ffn_union_f16");
}
int ffn_union_down(const void * down_t_f16, int ff, int cols, int T, const void * scratch, const void * h_f16, float * const * parts, const float * add1, const float * add2, float * out, pi_stream_t stream) {
    static const int raised = raise_lds(ffn_union_down_kernel, kGwLds);
    if (raised != PI_OK) return raised;
    const UnionScratch at(ff, T);
    const int32_t * list = (const int32_t *)((const unsigned char *)scratch + at.list), * count = (const int32_t *)((const unsigned char *)scratch + at.count);
    hipStream_t st = (hipStream_t)stream;
    DownProduct d{(const __half *)down_t_f16, (const __half *)h_f16, list, add1, add2, out, cols, T, (uint32_t)(cols * 2), parts ? ff / kGtBK : 0, {}, 0, 0};
    for (int k = 0; parts && k < kUnionParts - 1; ++k) d.parts[k] = parts[k];
    hipLaunchKernelGGL(ffn_union_down_kernel, dim3(kUnionGrid), dim3(512), kGwLds, st, d, count);
    int shared = 0;                                                      // units of an XCD that were
    bool turns = false;                                                  // (or may be, by how many are listed)
    for (int x = 0; x < 8; ++x) {
        const DownSplit deal(DownDeal(cols, (T + kGwN - 1) / kGwN, parts != nullptr, x, 0, kUnionGrid / 8), d.most, d.most);
        turns = turns || deal.turns;
        if (deal.parts > 1) shared = std::max(shared, deal.deal.rest);
    }
    if (shared) hipLaunchKernelGGL(ffn_union_sum_kernel, dim3(kGwN / 4, shared, 8), dim3(256), 0, st, d, turns ? count : nullptr);
    return check_launch("pi_k_ffn_union_f16");
}
}  // namespace pi
extern "C" {

int pi_k_ffn_union_f16(const void * fc2_f16, int rank, const void * hid_f16, const void * up_f16, const void * gate_f16, const void * down_t_f16, int ff, int cols, const void * xn_f16, int T,
                       float threshold, void * scratch, void * h_f16, float * const * parts, const float * add1, const float * add2, float * out, int32_t * n_active, pi_stream_t stream) {
    if (!down_t_f16 || !add1 || !out) return pi::fail(PI_E_ARG, "pi_k_ffn_union_f16: bad arguments");
    if ((((uintptr_t)down_t_f16 | (uintptr_t)add1 | (uintptr_t)add2 | (uintptr_t)out) & 15) != 0) return pi::fail(PI_E_ARG, "pi_k_ffn_union_f16: operands must be 16-byte aligned");
    for (int k = 0; parts && k < kUnionParts - 1; ++k)                  // (stored to and read in pieces of 16 bytes)
        if (!parts[k] || ((uintptr_t)parts[k] & 15) != 0) return pi::fail(PI_E_ARG, "pi_k_ffn_union_f16: parts must be three buffers on 16 bytes");
    const int rc = pi::ffn_union_hidden(fc2_f16, rank, hid_f16, up_f16, gate_f16, ff, cols, xn_f16, T, threshold, scratch, h_f16, n_active, pi::HostAsk{}, stream);
    return rc != PI_OK ? rc : pi::ffn_union_down(down_t_f16, ff, cols, T, scratch, h_f16, parts, add1, add2, out, stream);
}

}  // extern "C"
