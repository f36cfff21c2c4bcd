// What the sparse FFN of a prompt chunk gives the large tiles of gemm_wide: the predictor's bits and the hidden vector under them.
#pragma once
#include "gemm_wide.hpp"

namespace {

// ffn_h_f16_kernel's values straight from the matrices, in the large tiles of gemm_wide: a tile holds 64 rows of up, the 64 rows of gate of the same neurons and
// twice that again (PAIRS), or 256 rows of up alone; a lane then holds both factors of its neurons, and neither of them (90 MB each
// for 2048 tokens of 11008 neurons) goes to memory.  The products' sums are formed in 32-column steps in fp32, as in the tiles of
// the dense mat-mul.  11008 x 4096 twice, us (two library products and ffn_h_f16_kernel before): 2047 tokens 675 -> 327 (1.13
// PFLOP/s), 1024 tokens 222 -> 174, 256 tokens 109 -> 61, 64 tokens 60 -> 46; 32768 x 8192 alone, 2047 tokens: 1100 -> 941.
// MASK: which neurons are active comes as bits (MaskProduct) instead of logits: a 16 x 16 tile's bit l of word r is its lane l's r-th neuron, as the
// accumulators lie.
// LIST: of the neurons in `list` alone, ff of them and their bits in that order (kernels_ffn_union.hip).
template <bool PAIRS, bool MASK, bool LIST = false> struct FfnProduct {
    static constexpr bool kPairs = PAIRS, kList = LIST, kTurned = false;
    static constexpr int kM = kGwM, kN = kGwN;
    __device__ __forceinline__ bool read_once(const WidePlace &) const { return false; }
    // Rows a multiple of 16 KB apart lie in few of the memory's channels: every 2048 of them begin at columns of their own (bits included, us, one place for all /
    // this: 32768 x 8192 alone, 17 tokens 124 / 94 and 128 135 / 104 (no bits), 129 tokens 161 / 142, 200 175 / 155, 400 247 / 252, 700 381 / 390, 2047 1027 / 1029; 4096 columns, twice 11008 rows: 129 tokens 63.2 /
    // 64.5, 2047 372 / 370, so not there).  The place goes by the row alone: a token's sums have one order
    // however many come along.  With LIST it is a row's place in the list, which the other tokens of the chunk decide.
    __device__ __forceinline__ int first(const WidePlace & p) const { return cols % 8192 ? 0 : p.row0 / 2048 % 8 * nk / 8; }
    const __half * up, * gate, * x; const float * logits; float thr; __half * h16;
    int ff, cols, T, nk;
    const unsigned long long * mask;
    const int32_t * list;
    // the neuron that row `lane` of the w-th 64 rows belongs to, and where a neuron's row starts
    __device__ __forceinline__ int entry(const WidePlace & p, int w, int lane) const { return list[min(PAIRS ? p.row0 / 2 + w / 2 * 64 + lane : p.row0 + w * 64 + lane, ff - 1)]; }
    __device__ __forceinline__ uint32_t off_entry(int n) const { return (uint32_t)n * (uint32_t)(cols * 2); }
    __device__ __forceinline__ WidePlace place(const WideDeal & deal, int c) const {
        WidePlace p;
        int ty;
        deal.unit(c, ty, p.row0, p.rows);
        p.grp = 0; p.lo = ty * kGwN; p.n = min(T - p.lo, kGwN);
        return p;
    }
    __device__ __forceinline__ const unsigned char * base_a(const WidePlace &, int w) const {           // (no choice between members: a product that is put together in the kernel would be kept in scratch memory, 332 us instead of 303)
        const ptrdiff_t apart = PAIRS ? (const unsigned char *)gate - (const unsigned char *)up : 0;
        return (const unsigned char *)up + (w & 1) * apart;
    }
    __device__ __forceinline__ const unsigned char * base_b(const WidePlace & p) const { return (const unsigned char *)(x + (size_t)p.lo * cols); }
    __device__ __forceinline__ uint32_t off_a(const WidePlace & p, int r) const { return (uint32_t)(PAIRS ? p.row0 / 2 + r / 128 * 64 + r % 64 : p.row0 + r) * (uint32_t)(cols * 2); }
    __device__ __forceinline__ size_t off_b(const WidePlace &, int r) const { return (size_t)r * cols * 2; }
    template <int MT> __device__ __forceinline__ void store(const WidePlace & p, int rb, int tb, const pi_f4 (&acc)[MT][4], unsigned char * turn, int lane) const {
        constexpr int MO = PAIRS ? MT / 2 : MT;
        asm volatile("" : "+v"(lane));                 // what follows is computed here, not kept in registers across the products
        const int i = lane & 15, q = lane >> 4, n0 = PAIRS ? p.row0 / 2 + rb / 128 * 64 + rb % 128 : p.row0 + rb;          // this wave's first neuron
        const int left = ff - n0;                      // (a multiple of 64: whole tiles of 16 neurons or none)
        float4 lg[MASK ? 1 : 2][MO];
        // the bits of all these tokens and neurons in one trip (16 words at a time through the scalar unit: 349 us where this takes 332, twice 11008 x 4096 by 2047 tokens): word 4 m + r of tokens 16 nn .. is the (4 MO nn + 4 m + r)-th of the wave's lanes
        constexpr int kLoads = MO > 4 ? MO / 4 : 1;
        uint2 words[MASK ? kLoads : 1];
        auto fetch = [&](int nn) {
            if constexpr (MASK) return;
            const float * l = logits + (size_t)(p.lo + min(tb + nn * 16 + i, p.n - 1)) * ff + n0 + 4 * q;
#pragma unroll
            for (int m = 0; m < MO; ++m) lg[nn & 1][m] = *reinterpret_cast<const float4 *>(l + (m * 16 < left ? m * 16 : 0));
        };
        if (left <= 0) return;
        if constexpr (MASK) {
#pragma unroll
            for (int k = 0; k < kLoads; ++k) {
                const int at = 64 * k + lane, w = at % (4 * MO), tile = min((p.lo + tb) / 16 + min(at / (4 * MO), 3), (T - 1) / 16);
                words[k] = reinterpret_cast<const uint2 *>(mask)[((size_t)tile * (ff / 16) + n0 / 16) * 4 + (4 * w < left ? w : w & 3)];
            }
        }
        fetch(0);
#pragma unroll
        for (int nn = 0; nn < 4; ++nn) {
            if (nn < 3) fetch(nn + 1);
            uint2 out[MO];
#pragma unroll
            for (int m = 0; m < MO; ++m) {
                const float4 lm = MASK ? float4{} : lg[MASK ? 0 : nn & 1][m];
                const float l[4] = {lm.x, lm.y, lm.z, lm.w};
                __half h[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float u = acc[m][nn][r], v = PAIRS ? __fmul_rn(fmaxf(acc[(m + MO) % MT][nn][r], 0.0f), u) : fmaxf(u, 0.0f);
                    bool on;
                    if constexpr (MASK) {
                        const uint2 w = words[(nn * 4 * MO + 4 * m + r) / 64];
                        const int at = (nn * 4 * MO + 4 * m + r) % 64;
                        on = __builtin_amdgcn_inverse_ballot_w64((unsigned long long)(uint32_t)__builtin_amdgcn_readlane(w.y, at) << 32 | (uint32_t)__builtin_amdgcn_readlane(w.x, at));
                    } else {
                        on = !(l[r] < thr);
                    }
                    h[r] = __float2half_rn(on ? v : 0.0f);
                }
                out[m] = __builtin_bit_cast(uint2, h);
            }
            __builtin_amdgcn_sched_barrier(0);
            store_turned<8>(out, turn, lane, [&](int t, int piece) -> void * {
                const int to = tb + nn * 16 + t;
                return to < p.n && piece * 8 < left ? h16 + (size_t)(p.lo + to) * ff + n0 + piece * 8 : nullptr;
            });
        }
    }
};
// The predictor's second product, of which that is all anybody reads: 2047 tokens of 11008 neurons are 2.8 MB of bits instead of 90 of logits, written here
// and read by the FFN's first half.  Four 7B-shaped layers, us, library product with logits and this: 2047 tokens 3829 -> 3696, 600 1692 -> 1665, 300 1318 ->
// 1285; 13B 400 tokens 1408 -> 1378, 40B 700 tokens 1550 -> 1531.
// any: (null: nobody asks) for 64 tokens at a time which neurons fire for one of them, a bit a neuron.
struct MaskProduct {
    static constexpr bool kPairs = false, kList = false, kTurned = false;
    static constexpr int kM = kGwM, kN = kGwN;
    __device__ __forceinline__ bool read_once(const WidePlace &) const { return false; }
    __device__ __forceinline__ int first(const WidePlace &) const { return 0; }
    const __half * W, * x; float thr; unsigned long long * mask;
    int rows, cols, T, nk;
    uint16_t * any;
    __device__ __forceinline__ WidePlace place(const WideDeal & deal, int c) const {
        WidePlace p;
        int ty;
        deal.unit(c, ty, p.row0, p.rows);
        p.grp = 0; p.lo = ty * kGwN; p.n = min(T - p.lo, kGwN);
        return p;
    }
    __device__ __forceinline__ const unsigned char * base_a(const WidePlace &, int) const { return (const unsigned char *)W; }
    __device__ __forceinline__ const unsigned char * base_b(const WidePlace & p) const { return (const unsigned char *)(x + (size_t)p.lo * cols); }
    __device__ __forceinline__ uint32_t off_a(const WidePlace & p, int r) const { return (uint32_t)(p.row0 + r) * (uint32_t)(cols * 2); }
    __device__ __forceinline__ size_t off_b(const WidePlace &, int r) const { return (size_t)r * cols * 2; }
    template <int MT> __device__ __forceinline__ void store(const WidePlace & p, int rb, int tb, const pi_f4 (&acc)[MT][4], unsigned char *, int lane) const {
        const int left = min(p.rows - rb, 16 * MT) / 16;             // (rows % 128 == 0: whole tiles)
        unsigned long long fires = 0;                                // lane 4 m + r: word r of tile m, of all these tokens
#pragma unroll
        for (int nn = 0; nn < 4; ++nn) {
            const int tile = (p.lo + tb) / 16 + nn;
            if (tile > (T - 1) / 16) break;
            unsigned long long mine = 0;                             // lane 4 m + r: word r of tile m
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const unsigned long long w0 = __ballot(!(acc[m][nn][0] < thr)), w1 = __ballot(!(acc[m][nn][1] < thr)), w2 = __ballot(!(acc[m][nn][2] < thr)), w3 = __ballot(!(acc[m][nn][3] < thr));
                const unsigned long long w = lane & 2 ? (lane & 1 ? w3 : w2) : lane & 1 ? w1 : w0;
                if (lane >> 2 == m) mine = w;
            }
            if (lane < 4 * left) mask[((size_t)tile * (rows / 16) + (p.row0 + rb) / 16) * 4 + lane] = mine;
            fires |= mine;
        }
        if (!any || tb >= p.n) return;
        uint32_t bits = 0;                                           // lane m: tile m's neurons
#pragma unroll
        for (int f = 0; f < 4; ++f) bits |= ((uint32_t)__ballot((fires >> 16 * f & 0xFFFF) != 0) >> (4 * lane & 31) & 15u) << 4 * f;
        if (lane < left) any[(size_t)((p.lo + tb) / 64) * (rows / 16) + (p.row0 + rb) / 16 + lane] = (uint16_t)bits;
    }
};

}  // namespace
