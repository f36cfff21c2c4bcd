// Mat-muls of Q4_0 prompt chunks straight from the blocks.
#include "kernels_common.hpp"

#include <algorithm>
#include <type_traits>

namespace {

// ---------------------------------------------------------------------------------------------------------------------------------
// y[t][row] = epi(W[row] . x[t]) for a Q4_0 matrix and fp16 tokens: the values (q - 8) * d rounded to fp16 that the expanding kernels write
// are formed on the way into the matrix cores instead.
// TRANS = false: W[rows][cols].  true: the down projection as stored, W[cols][rows] with blocks of 32 rows of y.
// A workgroup has 16 MT rows.  Up to MT waves expand: of each stage of 256 columns, brought to registers three stages ahead, a lane takes two
// blocks of a row (TRANS: four bytes of a block in eight columns) and leaves its fp16 values in LDS as the matrix cores' fragments, once
// for the WN waves that multiply, each with 16 NT tokens of its own.  Those read the tokens' fragments, a KB in a row in the operand
// layout, straight to registers up to a stage ahead: each is used by one wave, and going through LDS would take more of its bandwidth than
// the weights do (with both operands copied to LDS and every wave expanding its own rows, 130 tokens of 12288 x 4096 took 33 us).
// A byte under 0x64 is 1024 + it in fp16, so q - 8 takes a permutation, a mask and one FMA for two (exact), and the product with d rounds
// once, as the float product of the expanding kernels does.
// The sums go over 32 columns a step in fp32, ascending, in parts of whole 128-column slabs, the longer ones first, that are added at the end: eight of a
// transposed matrix, two of one with more than twice as many rows as columns, at every length and in every tile.  More parts round less:
// relative error against 64 bits in one / two / four / eight parts, 130 tokens: 4096 x 4096 and 12288 x 4096 4.1e-7 / 2.9e-7 / 2.1e-7 / 1.6e-7,
// 32768 x 8192 5.7e-7 / 4.1e-7 / 2.9e-7 / 2.1e-7, 4096 x 11008 transposed 5.9e-7 / 4.1e-7 / 3.0e-7 / 2.2e-7, 8192 x 32768 1.02e-6 / 7.2e-7 /
// 5.1e-7 / 3.6e-7; expanded and multiplied by the library 4.1e-7, 5.7e-7, 5.9e-7 and 6.2e-7.  The longest sums, of the transposed
// matrices, have the most; one part would be enough elsewhere, and two are kept where results have them: another order of sums rounds
// activations to eight bits the other way here and there, which moves a model's logits by 1e-2.
// Of few tokens of a transposed matrix, which has few row tiles, 32 rows a workgroup leave most of each line of 128 bytes to other workgroups and read the
// tokens 128 times; four workgroups then share a tile of 64 rows, two parts of the sum each (kCqSlices).
// What bounds it at 130 tokens of 12288 x 4096 (21 us; the blocks alone 5, the matrix instructions 6): about 12 us are launch, first
// trip and last stores, which one workgroup a unit does not overlap with its products; the rest is shared about evenly between the
// tokens' way from the L2 (270 MB), expanding and multiplying.
// ---------------------------------------------------------------------------------------------------------------------------------
constexpr int kCqBK = 256, kCqSteps = kCqBK / 32;

__device__ __forceinline__ uint32_t cq_mul(uint32_t q, uint32_t mul, uint32_t add, uint32_t d) {       // two values: (q * mul + add) * d
    const __half2 v = __hfma2(__builtin_bit_cast(__half2, q), __builtin_bit_cast(__half2, mul), __builtin_bit_cast(__half2, add));
    return __builtin_bit_cast(uint32_t, __hmul2(v, __builtin_bit_cast(__half2, d)));
}
// low nibbles: 1024 + q, times 1, minus 1032; high ones: 1024 + 16 q, times 1 / 16, minus 72
__device__ __forceinline__ uint32_t cq_low(uint32_t q, uint32_t d) { return cq_mul((q & 0x000F000Fu) | 0x64006400u, 0x3C003C00u, 0xE408E408u, d); }
__device__ __forceinline__ uint32_t cq_high(uint32_t q, uint32_t d) { return cq_mul((q & 0x00F000F0u) | 0x64006400u, 0x2C002C00u, 0xD480D480u, d); }
typedef uint32_t cq_words __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t cq_pair __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kCqSlices = 4, kCqBufs = 2 * (kCqSlices - 1);
// slices (transposed, eight parts): 1, or kCqSlices workgroups of a tile with two parts each: the first one leaves their sum in y, the others leave theirs
// one by one in bufs, and chunk_parts_kernel adds them in the order of one workgroup
struct ChunkQ4 { const unsigned char * W; const unsigned char * x; int T, rows, cols, nx, ny, parts, epi; const float * add1, * add2; float * y; int slices; float * bufs[kCqBufs]; };

constexpr int cq_units(int MT, bool trans) { return !trans && MT > 4 ? 2 : 1; }          // pairs of blocks a lane expands of a stage
constexpr int cq_expand(int MT, bool trans) { return MT / cq_units(MT, trans); }            // expanding waves (TRANS: of one of two sets)
constexpr int cq_sets(int MT, bool trans) { return trans && MT == 2 ? 2 : 1; }
constexpr int cq_threads(int MT, int WN, bool trans) { return 64 * (cq_sets(MT, trans) * cq_expand(MT, trans) + WN); }
template <int MT, int NT, int WN, bool TRANS>
__global__ __launch_bounds__(cq_threads(MT, WN, TRANS), 2) void gemm_q4_chunk_kernel(ChunkQ4 a) {
    constexpr int kFrag = 1024, kStage = kCqSteps * MT * kFrag;
    extern __shared__ __align__(16) unsigned char smem[];           // [2][step][m][lane]: fragments
    // workgroup -> (row tile, token tile): an XCD takes row tiles that lie together and walks each one's token tiles in turn (one trip of W to its
    // L2; with TRANS a line of W holds the blocks of seven 32-row tiles)
    const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8, per = (a.nx + 7) / 8, tx = xcd * per + slot / a.ny, ty = slot % a.ny;
    if (tx >= a.nx) return;                                         // (slot / ny < per: the grid is 8 per ny)
    const int row0 = tx * 16 * MT, slabs = a.cols / 128;
    int nk = a.cols / kCqBK, k0 = 0, part = 0, until = a.parts;
    const auto slabs_ahead = [&](int p) { return p * (slabs / a.parts) + std::min(p, slabs % a.parts); };      // of the parts ahead of p (the longer parts come first)
    if (TRANS && a.slices > 1) {
        part = 2 * (int)blockIdx.y; until = part + 2;
        k0 = slabs_ahead(part) / 2; nk = slabs_ahead(until) / 2 - k0;   // (an even number of slabs)
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    // where a fragment's piece of row i and columns 8 g .. lies: rows trade places so that an expanding wave's stores spread over the banks
    auto place = [](int s, int m, int gg, int ii) {
        const int turn = !TRANS ? 4 * (s >> 1) : MT == 2 ? gg : (m >> 1) | (gg & 1) << 1;
        return ((s * MT + m) * 64 + gg * 16 + (ii ^ turn)) * 16;
    };
    if (wave >= WN) {
        constexpr int kUnits = cq_units(MT, TRANS), kWaves = cq_expand(MT, TRANS);
        const int w = wave - WN, set = w / kWaves, u = w % kWaves * 64 + lane;
        const int last = nk - 1;                                    // past it the last stage is fetched again, and expanded where nobody reads
        if constexpr (!TRANS) {
            // two blocks, nine words: d0 q0 .. q15 d1 q0 .. q15 in halves of words
            struct Raw { cq_words w[2]; uint32_t last; };
            struct Stage { Raw r[kUnits]; } held[3];
            const int pair = u & 3;
            uint32_t at[kUnits];                                    // (rows past the end are not stored)
            const size_t line = (size_t)a.cols / 32 * 18;
#pragma unroll
            for (int j = 0; j < kUnits; ++j) at[j] = (uint32_t)(std::min((u >> 2) + 16 * kWaves * j, a.rows - 1 - row0) * line) + pair * 36;
            auto fetch = [&](Stage & r, int k) {
                const unsigned char * p = a.W + row0 * line + (size_t)k * (kCqBK / 32 * 18);
#pragma unroll
                for (int j = 0; j < kUnits; ++j) {
                    const unsigned char * q = p + at[j];
                    r.r[j].w[0] = reinterpret_cast<const cq_words *>(q)[0]; r.r[j].w[1] = reinterpret_cast<const cq_words *>(q)[1];
                    r.r[j].last = reinterpret_cast<const uint32_t *>(q)[8];
                }
            };
            auto expand = [&](const Stage & st, unsigned char * to) {
#pragma unroll
                for (int j = 0; j < kUnits; ++j) {
                    const Raw & r = st.r[j];
                    const int row = (u >> 2) + 16 * kWaves * j;
                    const uint32_t D[9] = {r.w[0].x, r.w[0].y, r.w[0].z, r.w[0].w, r.w[1].x, r.w[1].y, r.w[1].z, r.w[1].w, r.last};
                    constexpr uint32_t lo = 0x0C010C00u, hi = 0x0C030C02u;
#pragma unroll
                    for (int blk = 0; blk < 2; ++blk) {
                        const uint32_t d = blk ? __builtin_amdgcn_perm(D[4], D[4], 0x03020302u) : __builtin_amdgcn_perm(D[0], D[0], 0x01000100u);
#pragma unroll
                        for (int h = 0; h < 2; ++h) {               // bytes 0 .. 7, then 8 .. 15
                            pi_u32x4 low, high;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int half = (blk ? 10 : 1) + 4 * h + e;      // of a word
                                const uint32_t q = __builtin_amdgcn_perm(D[half >> 1], D[half >> 1], half & 1 ? hi : lo);
                                low[e] = cq_low(q, d); high[e] = cq_high(q, d);
                            }
                            *reinterpret_cast<pi_u32x4 *>(to + place(2 * pair + blk, row >> 4, h, row & 15)) = low;
                            *reinterpret_cast<pi_u32x4 *>(to + place(2 * pair + blk, row >> 4, 2 + h, row & 15)) = high;
                        }
                    }
                }
            };
#pragma unroll
            for (int r = 0; r < 3; ++r) fetch(held[r], std::min(r, last));
            expand(held[0], smem);
            fetch(held[0], std::min(3, last));
            __syncthreads();
            for (int k = 0; k < nk; k += 3) {
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    if (k + r >= nk) break;
                    expand(held[(r + 1) % 3], smem + ((k + r + 1) & 1) * kStage);
                    fetch(held[(r + 1) % 3], std::min(k + r + 4, last));
                    __syncthreads();
                }
            }
        } else {
            // four bytes of eight columns: rows 4 cw .. 4 cw + 3 (low nibbles) and those 16 behind (high)
            // (blocks start on 2 bytes: a lane reads the two whole words around its four bytes, words of the block or of the one ahead; the
            // first of its four lanes then has the scale as well.  What bounds this are the lines of 128 bytes that 18 or 36 are taken of)
            struct Raw { cq_pair q[8]; } held[3];
            const int cw = u & 3, blk = MT == 2 ? 0 : (u >> 2) & 1, ng = MT == 2 ? u >> 2 : u >> 3;
            const size_t line = (size_t)a.rows / 32 * 18;
            const int block = row0 / 32 + blk;
            const uint32_t at = (uint32_t)(8 * ng * line) + block * 18, at_q = at + 4 * cw - (block & 1) * 2;
            const uint32_t mid = block & 1 ? 0x07060504u : 0x05040302u, scale = block & 1 ? 0x07060302u : 0x05040100u;
            auto fetch = [&](Raw & r, int k) {
                const unsigned char * p = a.W + (size_t)(k0 + k) * kCqBK * line;
#pragma unroll
                for (int e = 0; e < 8; ++e) r.q[e] = *reinterpret_cast<const cq_pair *>(p + e * line + at_q);
            };
            pi_u32x4 low[4], high[4];
            auto expand = [&](const Raw & r) {
                uint32_t d[4], w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) w[e] = __builtin_amdgcn_perm(r.q[e].y, r.q[e].x, mid);
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = (uint32_t)pi_dpp_i32<0x00, 0xF>((int)__builtin_amdgcn_perm(r.q[2 * e + 1].x, r.q[2 * e].x, scale));
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t q = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], 0x0C040C00u + 0x00010001u * b);
                        low[b][e] = cq_low(q, d[e]); high[b][e] = cq_high(q, d[e]);
                    }
            };
            auto put = [&](unsigned char * to) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    *reinterpret_cast<pi_u32x4 *>(to + place(ng >> 2, 2 * blk, ng & 3, 4 * cw + b)) = low[b];
                    *reinterpret_cast<pi_u32x4 *>(to + place(ng >> 2, 2 * blk + 1, ng & 3, 4 * cw + b)) = high[b];
                }
            };
            if constexpr (cq_sets(MT, TRANS) == 1) {
#pragma unroll
                for (int r = 0; r < 3; ++r) fetch(held[r], std::min(r, last));
                expand(held[0]);
                put(smem);
                fetch(held[0], std::min(3, last));
                __syncthreads();
                for (int k = 0; k < nk; k += 3) {
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        if (k + r >= nk) break;
                        expand(held[(r + 1) % 3]);
                        put(smem + ((k + r + 1) & 1) * kStage);
                        fetch(held[(r + 1) % 3], std::min(k + r + 4, last));
                        __syncthreads();
                    }
                }
                return;
            }
            // two sets of waves, one for the even stages and one for the odd ones: a stage is expanded while the one two ahead of it is
            // multiplied and stored during the next
            fetch(held[0], std::min(set, last));
            fetch(held[1], std::min(set + 2, last));
            expand(held[0]);
            fetch(held[0], std::min(set + 4, last));
            if (set == 0) { put(smem); expand(held[1]); fetch(held[1], std::min(6, last)); }
            __syncthreads();
            // what a set does in turn, from stage k0 on: put its expanded stage (k + 1), then expand the next one of its own
            int k = 0;
            if (set == 1) { put(smem + kStage); __syncthreads(); k = 1; }
            for (; k < nk; k += 4) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const int j = k + 2 * r;                        // stage j is multiplied; this set's next is j + 2
                    if (j >= nk) break;
                    if (!(set == 0 && j == 0)) { expand(held[(r + 1) & 1]); fetch(held[(r + 1) & 1], std::min(j + 6, last)); }
                    __syncthreads();
                    if (j + 1 >= nk) break;
                    put(smem + (j & 1) * kStage);
                    __syncthreads();
                }
            }
        }
        return;
    }
    pi_f4 acc[MT][NT], sum[MT][NT];                                 // of the parts that are done, and of the present one
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = sum[m][n] = pi_f4{0.0f, 0.0f, 0.0f, 0.0f};
    int left = slabs / a.parts + (part < slabs % a.parts ? 1 : 0);  // slabs of 128 columns left of the present part
    auto fold = [&]() {
        if (TRANS && blockIdx.y > 0 && part + 1 == until) return;      // (the second part of a slice behind the first stays by itself)
        left = slabs / a.parts + (++part < slabs % a.parts ? 1 : 0);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[m][n][r] += sum[m][n][r];
                sum[m][n] = pi_f4{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };
    const int tile0 = (ty * WN + wave) * NT, tiles = (a.T + 15) / 16;
    const unsigned char * xt[NT];                                   // (tiles past the end read the last one and are not stored)
#pragma unroll
    for (int n = 0; n < NT; ++n) xt[n] = a.x + (size_t)std::min(tile0 + n, tiles - 1) * 32 * a.cols + (size_t)k0 * (kCqSteps * kFrag) + lane * 16;
    // steps ahead a token's fragments are requested: a stage where the registers hold that many
    constexpr int kRegs = cq_threads(MT, WN, TRANS) > 512 ? 168 : 256, kHeld = MT * NT * 8 + MT * 8 + 44;
    constexpr int kRing = kHeld + NT * 32 <= kRegs ? kCqSteps : kHeld + NT * 16 <= kRegs ? kCqSteps / 2 : kCqSteps / 4;
    pi_u32x4 fb[kRing][NT], fa[4][MT];
    auto tokens = [&](int k, int s) {
#pragma unroll
        for (int n = 0; n < NT; ++n) fb[s % kRing][n] = pi_ld16(xt[n] + (size_t)k * (kCqSteps * kFrag) + s * kFrag);
    };
    auto weights = [&](int k, int s) {
#pragma unroll
        for (int m = 0; m < MT; ++m) fa[s & 3][m] = *reinterpret_cast<const pi_u32x4 *>(smem + (k & 1) * kStage + place(s, m, g, i));
    };
#pragma unroll
    for (int s = 0; s < kRing; ++s) tokens(0, s);
    constexpr int kAhead = MT * NT >= 6 ? 1 : 2;                    // steps of MFMAs between a fragment's request and its use
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kAhead; ++s) weights(0, s);
    for (int k = 0; k < nk; ++k) {
#pragma unroll
        for (int s = 0; s < kCqSteps; ++s) {
            __builtin_amdgcn_sched_barrier(0);
            if (s == kCqSteps - kAhead) __syncthreads();            // the next stage is whole, and this one has been read
            if (s < kCqSteps - kAhead) weights(k, s + kAhead);
            else weights(k + 1, s + kAhead - kCqSteps);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) sum[m][n] = mma16<__half>(fa[s & 3][m], fb[s % kRing][n], sum[m][n]);
            if (s + kRing < kCqSteps) tokens(k, s + kRing);
            else tokens(std::min(k + 1, nk - 1), s + kRing - kCqSteps);
            if (s % 4 == 3 && --left == 0) fold();
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int row = row0 + m * 16 + 4 * g, tok = (tile0 + n) * 16 + i;
            if (tok >= a.T || row >= a.rows) continue;              // (rows % 4 == 0)
            const size_t o = (size_t)tok * a.rows + row;
            float v[4] = {acc[m][n][0], acc[m][n][1], acc[m][n][2], acc[m][n][3]};
            if (TRANS && a.slices > 1) {
                float * to = blockIdx.y ? a.bufs[2 * blockIdx.y - 2] : a.y;
                *reinterpret_cast<float4 *>(to + o) = make_float4(v[0], v[1], v[2], v[3]);
                if (blockIdx.y) *reinterpret_cast<float4 *>(a.bufs[2 * blockIdx.y - 1] + o) = make_float4(sum[m][n][0], sum[m][n][1], sum[m][n][2], sum[m][n][3]);
                continue;
            }
            if (a.epi == PI_EPI_RELU) { for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.0f); }
            else if (a.epi >= PI_EPI_ADD) {
                const float4 a1 = *reinterpret_cast<const float4 *>(a.add1 + o);
                v[0] = __fadd_rn(v[0], a1.x); v[1] = __fadd_rn(v[1], a1.y); v[2] = __fadd_rn(v[2], a1.z); v[3] = __fadd_rn(v[3], a1.w);
                if (a.epi == PI_EPI_ADD2) {
                    const float4 a2 = *reinterpret_cast<const float4 *>(a.add2 + o);
                    v[0] = __fadd_rn(v[0], a2.x); v[1] = __fadd_rn(v[1], a2.y); v[2] = __fadd_rn(v[2], a2.z); v[3] = __fadd_rn(v[3], a2.w);
                }
            }
            *reinterpret_cast<float4 *>(a.y + o) = make_float4(v[0], v[1], v[2], v[3]);
        }
}

__global__ __launch_bounds__(256) void chunk_parts_kernel(ChunkQ4 a) {
    const size_t o = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (o >= (size_t)a.T * a.rows) return;
    float4 v = *reinterpret_cast<const float4 *>(a.y + o), b[kCqBufs], a1 = make_float4(0, 0, 0, 0), a2 = a1;
#pragma unroll
    for (int k = 0; k < kCqBufs; ++k) b[k] = *reinterpret_cast<const float4 *>(a.bufs[k] + o);
    if (a.epi >= PI_EPI_ADD) a1 = *reinterpret_cast<const float4 *>(a.add1 + o);
    if (a.epi == PI_EPI_ADD2) a2 = *reinterpret_cast<const float4 *>(a.add2 + o);
#pragma unroll
    for (int k = 0; k < kCqBufs; ++k) { v.x += b[k].x; v.y += b[k].y; v.z += b[k].z; v.w += b[k].w; }
    if (a.epi == PI_EPI_RELU) v = make_float4(fmaxf(v.x, 0.0f), fmaxf(v.y, 0.0f), fmaxf(v.z, 0.0f), fmaxf(v.w, 0.0f));
    if (a.epi >= PI_EPI_ADD) v = make_float4(__fadd_rn(v.x, a1.x), __fadd_rn(v.y, a1.y), __fadd_rn(v.z, a1.z), __fadd_rn(v.w, a1.w));
    if (a.epi == PI_EPI_ADD2) v = make_float4(__fadd_rn(v.x, a2.x), __fadd_rn(v.y, a2.y), __fadd_rn(v.z, a2.z), __fadd_rn(v.w, a2.w));
    *reinterpret_cast<float4 *>(a.y + o) = v;
}

template <int MT, int NT, int WN, bool TRANS> int launch_chunk_q4(ChunkQ4 a, hipStream_t st) {
    constexpr size_t lds = (size_t)2 * kCqSteps * MT * 1024;
    a.nx = (a.rows + 16 * MT - 1) / (16 * MT); a.ny = ((a.T + 15) / 16 + NT * WN - 1) / (NT * WN);
    if constexpr (lds > 64 * 1024) {
        static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_q4_chunk_kernel<MT, NT, WN, TRANS>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (raised != hipSuccess) return pi::hip_fail(raised, "pi_k_gemm_q4_chunk: LDS size");
    }
    hipLaunchKernelGGL((gemm_q4_chunk_kernel<MT, NT, WN, TRANS>), dim3((unsigned)(8 * ((a.nx + 7) / 8) * a.ny), a.slices), dim3(cq_threads(MT, WN, TRANS)), lds, st, a);
    return pi::check_launch("pi_k_gemm_q4_chunk");
}

// Tiles as 100 * (16-row tiles) + 10 * (16-token tiles a wave) + waves
// (no 96 rows with three token tiles for each of four waves: one round of that takes as long as two of 333 or 334, two workgroups of which share a
// unit.  17 to 24 token tiles of 7B shapes: 11008 x 4096, us, 280 tokens 53.3 / 36.7, 360 tokens 55.0 / 42.2; 12288 x 4096 54.3 / 39.9)
constexpr int kCqTiles[] = {112, 122, 123, 215, 232, 314, 323, 333, 334, 414, 423, 424, 434, 444, 624};
constexpr int kCqTilesT[] = {212, 213, 215, 223, 422, 423, 424, 433, 434};
// What a launch takes goes with the rounds of workgroups over the compute units times what 32 columns of a tile take of a unit, in clocks: the
// tokens' fragments at 64 bytes a clock, the matrix instructions of a SIMD, or the latency of a step where both are little; transposed, the
// lines of 128 bytes that 18 or 36 are taken of, and the tokens.  Of 152 measured launches (19 lengths of 17 .. 512 tokens, the matrices of 7B
// and 13B shapes) the choice is within 10 % of the fastest in 150 and 12 % slower in the worst, 0.4 % on average.
int cq_choose(int rows, int T, bool trans, int units) {
    const int * tiles = trans ? kCqTilesT : kCqTiles, n = trans ? (int)(sizeof kCqTilesT / sizeof(int)) : (int)(sizeof kCqTiles / sizeof(int));
    int best = tiles[0];
    double least = 1e30;
    for (int j = 0; j < n; ++j) {
        const int m = tiles[j] / 100, t = tiles[j] / 10 % 10, w = tiles[j] % 10;
        const long long groups = (long long)((rows + 16 * m - 1) / (16 * m)) * (((T + 15) / 16 + t * w - 1) / (t * w));
        const double step = trans ? (m == 2 ? 100.0 + 12.0 * t * w : 180.0 + 13.0 * t * w) : std::max({16.0 * t * w + 4.5 * m, 18.4 * m * t * ((w + 3) / 4), 110.0}) + 40.0;
        const double c = (double)((groups + units - 1) / units) * step;
        if (c < least) { least = c; best = tiles[j]; }
    }
    return best;
}

// Whether the transposed product is done in slices, by what both ways take in clocks: rounds of workgroups over the units times the steps of one and what a
// round takes by itself (with 32 rows also the lines of every row tile, which all token tiles share), and of slices a launch and 36 bytes a value more.
// Over 80 launches (17 .. 512 tokens of 2048 x 5632, 4096 x 11008, 4096 x 16384, 5120 x 13824 and 8192 x 32768) slices take 0.84 of what one
// workgroup a tile does on average and never more.  us, one and slices: 4096 x 11008, 17 tokens 25.6 / 19.5, 130 36.6 / 28.0, 192 40.9 / 33.2, 288 55.9 /
// 50.5, 333 54.9 / 60.0 (not taken); 5120 x 13824, 130 tokens 55.0 / 47.8; 8192 x 32768, 64 tokens 113 / 73.
double cq_clocks(int tile, int rows, int cols, int T, int slices, int units) {
    const int m = tile / 100, t = tile / 10 % 10, w = tile % 10, nx = (rows + 16 * m - 1) / (16 * m);
    const long long groups = (long long)nx * (((T + 15) / 16 + t * w - 1) / (t * w)) * slices;
    const double step = m == 2 ? std::max(100.0 + 12.0 * t * w, 150.0 * std::min(1.0, (double)nx * slices / units)) : 180.0 + 13.0 * t * w;
    return (double)((groups + units - 1) / units) * (step * cols / 32 / slices + (m == 2 ? 6000.0 : 4000.0)) + (slices > 1 ? 4600.0 + 0.018 * T * rows : 0.0);
}
int cq_slices(int & tile, int rows, int cols, int T, int units) {
    int best = tile, slices = 1;
    double least = cq_clocks(tile, rows, cols, T, 1, units);
    for (int t : kCqTilesT) {
        const double c = cq_clocks(t, rows, cols, T, kCqSlices, units);
        if (c < least) { least = c; best = t; slices = kCqSlices; }
    }
    tile = best;
    return slices;
}

}  // namespace

extern "C" {

int pi_k_gemm_q4_chunk_supported(int rows, int cols) { return rows > 0 && cols > 0 && rows % 64 == 0 && cols % kCqBK == 0 && (long long)rows * cols < (1LL << 31); }

int pi_k_gemm_q4_chunk(const void * W_q4, int rows, int cols, int transposed, const void * x_ol, int T, int epilogue, const float * add1, const float * add2,
                       float * y, int tile, pi_stream_t stream) {
    return pi_k_gemm_q4_chunk_parts(W_q4, rows, cols, transposed, x_ol, T, epilogue, add1, add2, y, tile, nullptr, stream);
}

int pi_k_gemm_q4_chunk_parts(const void * W_q4, int rows, int cols, int transposed, const void * x_ol, int T, int epilogue, const float * add1, const float * add2,
                             float * y, int tile, float * const * bufs, pi_stream_t stream) {
    if (!W_q4 || !x_ol || !y || T <= 0) return pi::fail(PI_E_ARG, "pi_k_gemm_q4_chunk: null pointer or empty shape");
    if (epilogue < 0 || epilogue > PI_EPI_ADD2 || (epilogue >= PI_EPI_ADD && !add1) || (epilogue == PI_EPI_ADD2 && !add2))
        return pi::fail(PI_E_ARG, "pi_k_gemm_q4_chunk: bad epilogue arguments");
    if (!pi_k_gemm_q4_chunk_supported(rows, cols) || (((uintptr_t)x_ol | (uintptr_t)y | (uintptr_t)add1 | (uintptr_t)add2) & 15) != 0 || ((uintptr_t)W_q4 & 3) != 0)
        return pi::fail(PI_E_UNSUPPORTED, "pi_k_gemm_q4_chunk: cols % 256 == 0, rows % 64 == 0, W on 4 bytes and the other operands on 16");
    if (T > 65536) return pi::fail(PI_E_UNSUPPORTED, "pi_k_gemm_q4_chunk: at most 65536 tokens");
    const int parts = transposed ? 8 : rows > 2 * cols ? 2 : 1;
    ChunkQ4 a{(const unsigned char *)W_q4, (const unsigned char *)x_ol, T, rows, cols, 0, 0, std::min(parts, cols / 128), epilogue, add1, add2, y, 1, {}};
    hipStream_t st = (hipStream_t)stream;
    bool room = bufs && transposed && a.parts == 2 * kCqSlices;
    for (int k = 0; room && k < kCqBufs; ++k) { a.bufs[k] = bufs[k]; room = bufs[k] && ((uintptr_t)bufs[k] & 15) == 0; }
    if (tile >= 1000) { if (!room) return pi::fail(PI_E_ARG, "pi_k_gemm_q4_chunk_parts: no room for parts"); tile -= 1000; a.slices = kCqSlices; }
    if (tile == 0) {
        const int units = pi::compute_units();
        if (units <= 0) return PI_E_HIP;
        tile = cq_choose(rows, T, transposed != 0, units);
        if (room) a.slices = cq_slices(tile, rows, cols, T, units);
    }
    const auto launch = [&]() -> int {
#define PI_CQ1(M, N, W) case M * 100 + N * 10 + W: return launch_chunk_q4<M, N, W, false>(a, st)
#define PI_CQ2(M, N, W) case M * 100 + N * 10 + W: return launch_chunk_q4<M, N, W, true>(a, st)
    if (!transposed) {
        switch (tile) {
            PI_CQ1(1, 1, 2); PI_CQ1(1, 2, 2); PI_CQ1(1, 2, 3); PI_CQ1(2, 1, 5); PI_CQ1(2, 3, 2); PI_CQ1(3, 1, 4); PI_CQ1(3, 2, 3); PI_CQ1(3, 3, 3);
            PI_CQ1(3, 3, 4); PI_CQ1(4, 1, 4); PI_CQ1(4, 2, 3); PI_CQ1(4, 2, 4); PI_CQ1(6, 2, 4); PI_CQ1(4, 3, 4); PI_CQ1(4, 4, 4);
        }
    } else {
        switch (tile) {
            PI_CQ2(2, 1, 2); PI_CQ2(2, 1, 3); PI_CQ2(2, 1, 5); PI_CQ2(2, 2, 3); PI_CQ2(4, 2, 2); PI_CQ2(4, 2, 3); PI_CQ2(4, 2, 4); PI_CQ2(4, 3, 3); PI_CQ2(4, 3, 4);
        }
    }
#undef PI_CQ1
#undef PI_CQ2
    return pi::fail(PI_E_ARG, "pi_k_gemm_q4_chunk: no such tile");
    };
    const int rc = launch();
    if (rc != PI_OK || a.slices == 1) return rc;
    hipLaunchKernelGGL(chunk_parts_kernel, dim3((unsigned)(((size_t)T * rows / 4 + 255) / 256)), dim3(256), 0, st, a);
    return pi::check_launch("pi_k_gemm_q4_chunk_parts");
}

}  // extern "C"
