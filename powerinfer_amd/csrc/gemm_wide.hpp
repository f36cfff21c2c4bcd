// The matrix-core product of long prompts in tiles of 256 rows x 128 tokens or 128 x 256, shared by the experts' products and the sparse FFN's.
#pragma once
#include "gemm_tile.hpp"

namespace {

// Sixteen rows by 32 columns of an operand that lies column by column in LDS, 512 bytes (256 rows) each: the matrix cores want eight consecutive columns of
// one row in a lane, which ds_read_b64_tr_b16 turns out of four columns of sixteen rows at a time.  A column's 32-byte pieces are stored at
// piece ^ turned_key(column): the eight columns that half a wave reads the same piece of fall on different banks.
__device__ __forceinline__ int turned_key(int column) { return (column & 3) | (column >> 3 & 1) << 2; }
__device__ __forceinline__ pi_u32x4 turned_fragment(const unsigned char * p) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 * ptr;
    union { s4 half[2]; pi_u32x4 whole; } f;
    f.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)p);
    f.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(p + 4 * 512));
    return f.whole;
}

// ---------------------------------------------------------------------------------------------------------------------------------
// One workgroup per compute unit that stays for all of its units.  Four waves multiply (128 x 64 outputs each), four copy: a stage of 64
// columns goes from memory straight to LDS, three stages deep and on into the next unit, and a copy that has to wait for the
// memory's queues holds up no matrix instruction (copying from the multiplying waves themselves: 238 us for the first product
// below).  A multiplying wave reads the fragments of a stage's second 32 columns under the products of the first and those of the
// next stage's first 32 under the products of the second, with the one barrier of a stage in between: behind it the next stage is
// whole and the present one is free to be copied over.  LDS rows and swizzle are GemmTile's; a copy's 64 lanes bring eight rows of
// 128 bytes and take the swizzle on the side they read from.  Where half a tile or less is wanted (half its rows, or so few tokens that a wave would
// have none) the four waves share that half, 64 x 64 outputs each.  The sums are formed in GemmTile's order: 32 columns a step, beginning at a stage that
// depends on the product and the row alone (first), so that a token's outputs are the same bits whichever tiles it falls into.  Not so over
// listed neurons: the list, where a row's sum begins and (kTurned) into which parts it is cut are the chunk's, by its length and by what all of its tokens fire.
// Measured (us; 128 x 128 tiles of GemmTile before): 64 experts of 192 tokens on average, 1408 x 4096: 301 -> 215, 4096 x 1408:
// 307 -> 226 (weights alone: 123 at 6 TB/s); one group of 12288: 199 -> 133, 1.07 PFLOP/s; 16 experts of 128: 51 -> 45 and 38 -> 34.
// ---------------------------------------------------------------------------------------------------------------------------------
constexpr int kGwM = 256, kGwN = 128, kGwStages = 3, kGwStage = (kGwM + kGwN) * kGtRow, kGwTurn = 2048, kGwLds = kGwStages * kGwStage + 128 + 4 * kGwTurn;

// token tiles of a band of one group's product (one by one, 2047 tokens by twice 11008 x 4096 take 424 us: 32 workgroups share a token tile and
// each its own rows; by 4 327, by 8 327, by 16 343)
constexpr int kGwBand = 8;
// The units of this workgroup: the products (token tile, 256 rows) are dealt out so that an XCD works through a contiguous range of them,
// band token tiles by row tiles (its L2 then serves a band's tokens and a few row tiles to all of its workgroups), the row tiles of more
// than 128 rows first, then the shorter ones, which take half the time.  What does not fill the XCD's
// workgroups once more at the end is cut into halves of a tile's rows if that gives no workgroup two of them.  (256 rows: `tile` of them.)
struct WideDeal {
    int rows, n_tiles, band, tile, nl, xcd, slot, slots, per_long, per_short, n_long, rounds, rest_unit, rest_row, count;
    bool halves;
    __device__ __forceinline__ WideDeal(int rows_, int n_tiles_, int band_, int tile_ = kGwM) {
        rows = rows_; n_tiles = n_tiles_; band = band_; tile = tile_;
        const int nx = (rows + tile - 1) / tile, last = rows - (nx - 1) * tile;
        nl = last > tile / 2 ? nx : nx - 1;
        xcd = (int)blockIdx.x % 8; slot = (int)blockIdx.x / 8; slots = (int)gridDim.x / 8;
        per_long = (n_tiles * nl + 7) / 8; per_short = nl < nx ? (n_tiles + 7) / 8 : 0;
        n_long = max(min(n_tiles * nl - xcd * per_long, per_long), 0);
        const int n = n_long + max(min(nl < nx ? n_tiles - xcd * per_short : 0, per_short), 0), rest = n % slots;
        rounds = n / slots;
        halves = rest > 0 && 2 * rest <= slots;
        rest_unit = rounds * slots + (halves ? slot / 2 : slot); rest_row = halves ? slot % 2 * (tile / 2) : 0;
        count = rounds + (slot < (halves ? 2 * rest : rest) && !(rest_row && rest_unit >= n_long) ? 1 : 0);
    }
    // the c-th of them: its token tile, its first row and how many there are
    __device__ __forceinline__ void unit(int c, int & ty, int & row0, int & n_rows) const {
        const int u = c < rounds ? c * slots + slot : rest_unit;
        if (u < n_long) {
            const int at = xcd * per_long + u, b0 = at / (band * nl) * band, high = min(band, n_tiles - b0), in = at - b0 * nl;
            ty = b0 + in % high; row0 = in / high * tile;
        } else {
            ty = xcd * per_short + u - n_long; row0 = (rows - 1) / tile * tile;
        }
        if (c >= rounds) row0 += rest_row;
        n_rows = min(rows - row0, c < rounds || !halves ? tile : tile / 2);
    }
};
inline unsigned wide_blocks(long long units) { return (unsigned)(units < 128 ? (2 * units + 7) / 8 * 8 : 256); }

struct WidePlace { int grp, lo, n, row0, rows; };       // of a unit: group, first token and tokens, first row and rows

// P (a product): nk stages of 64 columns; place(deal, c); base_a(p, w), base_b(p): where the rows of a tile's w-th 64 rows and its tokens start, and
// off_a(p, r), off_b(p, r): the bytes from there to tile row and token r (in range: r is cut to the unit's); kPairs: a wave's rows
// are two runs of MT / 2 tiles, `gap` rows apart beyond their own where MT is 4; read_once(p): no other unit reads these rows of W; first(p): the column stage a unit begins with, which may depend on nothing
// but its group and rows; kM, kN: the tile; kList: a tile's rows are not consecutive: entry(p, w, lane) says which the w-th 64 are and off_entry where
// one starts; kTurned: W lies with its rows along the contiguous dimension, and the column of it that a product's column c is stands in turned[c]
// (col_bytes from one to the next, base_a(p, w) is the tile's place in column 0; M 256, columns multiples of 64), and a unit may have a part of the stages: stages(p)
// of them from first(p) on; store<MT>(p, rb, tb, acc, turn, lane): the
// outputs of rows rb .. and tokens tb .. of the tile.
template <typename EL, typename P, typename D> __device__ __forceinline__ void gemm_wide(const P & prod, const D & deal, unsigned char * smem) {
    if (deal.count == 0) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    constexpr int M = P::kM, N = P::kN, CA = M / 32, CB = N / 32;   // rows and tokens of a tile, copies of a wave a stage (twelve)
    static_assert(CA + CB == 12, "the waits below count them");
    const int count = deal.count;
    const auto stages = [&](const WidePlace & p) { if constexpr (P::kTurned) return prod.stages(p); else return prod.nk; };
    WidePlace * places = reinterpret_cast<WidePlace *>(smem + kGwStages * kGwStage);      // of this unit and those behind it, written by the first copying wave
    if (wave >= 4) {
        // A wave that copies.  Of each stage CA times eight rows of W and CB times eight of x are its own, each 128 bytes; lane l brings
        // the piece that belongs at place l % 8 of row l / 8
        const int w = wave - 4, piece = ((lane & 7) ^ (lane >> 3)) * 16;
        uint32_t va[CA];                                            // (kTurned: the pieces of a column, by two bits of its number)
        size_t vb[CB];
        const unsigned char * fa, * fb;
        int k = 0, c = 0, first = 0, nk = prod.nk;                                // a unit's stages are copied from column stage `first` on, around the end
        bool once = false;
        int entry = 0;
        if constexpr (P::kList) { static_assert(M == 256, "a wave's entries are 64"); entry = prod.entry(prod.place(deal, 0), w, lane); }
        auto aim = [&]() {
            const WidePlace p = prod.place(deal, c);
            if (w == 0 && lane == 0) places[c & 3] = p;
            ++c;
            fa = prod.base_a(p, w); fb = prod.base_b(p); once = prod.read_once(p); first = prod.first(p); nk = stages(p);
            if constexpr (P::kList) {
#pragma unroll
                for (int j = 0; j < CA; ++j) va[j] = prod.off_entry(__shfl(entry, 8 * j + (lane >> 3))) + piece;
                entry = prod.entry(prod.place(deal, min(c, count - 1)), w, lane);      // a unit ahead: nothing waits for them but what is older anyway
            } else if constexpr (P::kTurned) {
#pragma unroll
                for (int j = 0; j < 4; ++j) va[j] = min(((lane >> 1 & 15) ^ turned_key(2 * (j & 1) + 8 * (j >> 1) + (lane >> 5))) * 32 + (lane & 1) * 16, p.rows * 2 - 16);
            } else {
#pragma unroll
                for (int j = 0; j < CA; ++j) va[j] = prod.off_a(p, min(8 * CA * w + 8 * j + (lane >> 3), p.rows - 1)) + piece;
            }
#pragma unroll
            for (int j = 0; j < CB; ++j) vb[j] = prod.off_b(p, min(8 * CB * w + 8 * j + (lane >> 3), p.n - 1)) + piece;
        };
        typedef const __attribute__((address_space(1))) void * gptr;
        typedef __attribute__((address_space(3))) void * lptr;
        auto copy_stage = [&](unsigned char * stage) {             // past the last unit the last stage is copied again, and not used
            const int ks = P::kTurned || first + k < nk ? first + k : first + k - nk;
            const size_t at = (size_t)ks * kGtRow;
            if constexpr (P::kTurned) {                            // columns 16 w .. of the stage, two a copy
                typedef const __attribute__((address_space(4))) int32_t * sptr;
                const sptr list = (sptr)(prod.turned + ks * kGtBK + 16 * w);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t o0 = (uint32_t)list[2 * j] * prod.col_bytes, o1 = (uint32_t)list[2 * j + 1] * prod.col_bytes;
                    __builtin_amdgcn_global_load_lds((gptr)(fa + ((lane & 32 ? o1 : o0) + va[(j & 1) | (j >> 2) << 1])), (lptr)(stage + (16 * w + 2 * j) * 512), 16, 0, 0);
                }
            } else if (once) {                                            // (the last operand of the builtin: 2 is the non-temporal hint)
#pragma unroll
                for (int j = 0; j < CA; ++j) __builtin_amdgcn_global_load_lds((gptr)(fa + at + va[j]), (lptr)(stage + 8 * (CA * w + j) * kGtRow), 16, 0, 2);
            } else {
#pragma unroll
                for (int j = 0; j < CA; ++j) __builtin_amdgcn_global_load_lds((gptr)(fa + at + va[j]), (lptr)(stage + 8 * (CA * w + j) * kGtRow), 16, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < CB; ++j) __builtin_amdgcn_global_load_lds((gptr)(fb + at + vb[j]), (lptr)(stage + (M + 8 * (CB * w + j)) * kGtRow), 16, 0, 0);
            if (++k < nk) return;
            if (c < count) { k = 0; aim(); } else k = nk - 1;
        };
        int total = count * nk;
        if constexpr (P::kTurned) { total = 0; for (int u = 0; u < count; ++u) total += stages(prod.place(deal, u)); }
        aim();
        for (int st = 0; st < kGwStages; ++st) copy_stage(smem + st * kGwStage);
        __builtin_amdgcn_s_waitcnt(0x4078);                         // vmcnt(24): the first stage; lgkmcnt(0): its place
        __builtin_amdgcn_s_barrier();
        for (int t = 0, cb = 0; t < total; ++t) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x007C);                     // vmcnt(12): the stage after t; lgkmcnt(0): a place
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            copy_stage(smem + cb * kGwStage);
            cb = cb == kGwStages - 1 ? 0 : cb + 1;
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);                         // vmcnt(0): no copy may arrive in LDS that is no longer this workgroup's
        return;
    }
    unsigned char * turn = smem + kGwStages * kGwStage + 128 + wave * kGwTurn;
    int cb = 0;                                                    // the stage that is being multiplied
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int koff[2] = {(q ^ (i & 7)) * 16, ((4 + q) ^ (i & 7)) * 16};
    auto run = [&](auto mt, const WidePlace & p, int rb, int tb) {  // rows rb .. and tokens tb .. of the tile are this wave's
        const int nk = stages(p);
        constexpr int MT = decltype(mt)::value, kGap = P::kPairs && MT == 4 ? 32 : 0;
        pi_f4 acc[MT][4];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] = pi_f4{0.0f, 0.0f, 0.0f, 0.0f};
        pi_u32x4 f0a[MT], f0b[4], f1a[MT], f1b[4];
        const int oa = (rb + i) * kGtRow, ob = (M + tb + i) * kGtRow;
        const int ot = (8 * q + (i >> 2)) * 512 + (i & 3) * 8, key = turned_key(8 * q + (i >> 2));
        auto ld = [&](int off) { return *reinterpret_cast<const pi_u32x4 *>(smem + cb * kGwStage + off); };
        auto lda = [&](int m, int h) {
            if constexpr (P::kTurned) return turned_fragment(smem + cb * kGwStage + ot + h * 32 * 512 + ((rb / 16 + m) ^ key) * 32);
            else return ld(oa + koff[h] + (m * 16 + (m >= MT / 2 ? kGap : 0)) * kGtRow);
        };
        auto ldb = [&](int n, int h) { return ld(ob + koff[h] + n * 16 * kGtRow); };
#pragma unroll
        for (int m = 0; m < MT; ++m) f0a[m] = lda(m, 0);
#pragma unroll
        for (int n = 0; n < 4; ++n) f0b[n] = ldb(n, 0);
        // a group: the four MFMAs of one fragment of W.  A phase's reads follow its first RD groups' MFMAs: they never stand before an MFMA
        // that waits for older ones, and the last groups cover their latency
        constexpr int RD = MT / 2, RA = MT / RD, RB = 4 / RD;
        for (int kt = 0; kt < nk; ++kt) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[m][n] = mma16<EL>(f0a[m], f0b[n], acc[m][n]);
                __builtin_amdgcn_sched_barrier(0);
                if (m < RD) {
#pragma unroll
                    for (int r = 0; r < RB; ++r) f1b[RB * m + r] = ldb(RB * m + r, 1);
#pragma unroll
                    for (int r = 0; r < RA; ++r) f1a[RA * m + r] = lda(RA * m + r, 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // the next stage has arrived (two more are on their way), and nobody reads this one any more
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F);                     // lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            cb = cb == kGwStages - 1 ? 0 : cb + 1;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[m][n] = mma16<EL>(f1a[m], f1b[n], acc[m][n]);
                __builtin_amdgcn_sched_barrier(0);
                if (m < RD) {
#pragma unroll
                    for (int r = 0; r < RB; ++r) f0b[RB * m + r] = ldb(RB * m + r, 0);
#pragma unroll
                    for (int r = 0; r < RA; ++r) f0a[RA * m + r] = lda(RA * m + r, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        prod.template store<MT>(p, rb, tb, acc, turn, lane);
    };
    auto idle = [&](const WidePlace & p) {                          // no tokens of this tile
        for (int kt = 0, nk = stages(p); kt < nk; ++kt) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            cb = cb == kGwStages - 1 ? 0 : cb + 1;
        }
        asm volatile("" ::: "memory");
    };
    for (int c = 0; c < count; ++c) {
        const int * pl = reinterpret_cast<const int *>(places + (c & 3));
        WidePlace p;
        p.grp = __builtin_amdgcn_readfirstlane(pl[0]); p.lo = __builtin_amdgcn_readfirstlane(pl[1]); p.n = __builtin_amdgcn_readfirstlane(pl[2]); p.row0 = __builtin_amdgcn_readfirstlane(pl[3]);
        p.rows = __builtin_amdgcn_readfirstlane(pl[4]);
        constexpr int kStep = P::kPairs ? 32 : 64;
        if constexpr (M == 128) {
            const bool half = p.rows <= 64, pairs = !half && p.n <= 128;
            const int tb = pairs ? 64 * (wave >> 1) : 64 * wave;
            if (tb >= p.n) idle(p);
            else if (half || pairs) run(std::integral_constant<int, 4>{}, p, pairs ? 64 * (wave & 1) : 0, tb);
            else run(std::integral_constant<int, 8>{}, p, 0, tb);
        } else if (p.rows <= 128) run(std::integral_constant<int, 4>{}, p, kStep * (wave & 1), 64 * (wave >> 1));
        else if (p.n <= 64) run(std::integral_constant<int, 4>{}, p, 128 * (wave >> 1) + kStep * (wave & 1), 0);
        else run(std::integral_constant<int, 8>{}, p, 128 * (wave & 1), 64 * (wave >> 1));
    }
}

// Outputs of 16 bits that come in whole pieces of 16 bytes leave through LDS: the lanes' quads of rows, stored as they are, are runs of 32 bytes a token
// (8 us for 256 x 128 outputs of a workgroup); eight tokens at a time, turned in 2 KB of the wave's own, leave in runs of up to
// 256 bytes.  out: what a lane holds of every 16 rows, PB bytes (8: four outputs of 16 bits, 4: two); to(t, piece): where 16 bytes of
// token t (of these sixteen) go, null: nowhere.
template <int PB, int MT, typename F> __device__ __forceinline__ void store_turned(const uint2 (&out)[MT], unsigned char * turn, int lane, F && to) {
    constexpr int kRow = MT * PB * 4, kPieces = kRow / 16, kToks = 64 / kPieces, kReads = (8 * kPieces + 63) / 64;      // bytes and pieces of a token, tokens a store takes
    const int i = lane & 15, q = lane >> 4, piece = lane % kPieces, first = lane / kPieces;
#pragma unroll
    for (int h = 0; h < 2; ++h) {                                   // tokens 0 .. 7 of the sixteen, then 8 .. 15
        unsigned char * mine = turn + (i & 7) * kRow;
        if ((i >> 3) == h) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if constexpr (PB == 4) *reinterpret_cast<uint32_t *>(mine + (m ^ (i & 7) % kPieces) * 16 + q * 4) = out[m].x;
                else *reinterpret_cast<uint2 *>(mine + ((2 * m + (q >> 1)) ^ ((i & 7) % kPieces)) * 16 + (q & 1) * 8) = out[m];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t0 = 0; t0 < kReads; ++t0) {
            const int t = t0 * kToks + first;
            const pi_u32x4 v = *reinterpret_cast<const pi_u32x4 *>(turn + (t & 7) * kRow + (piece ^ ((t & 7) % kPieces)) * 16);
            void * dst = t < 8 ? to(8 * h + t, piece) : nullptr;
            if (dst) *reinterpret_cast<pi_u32x4 *>(dst) = v;
        }
    }
}

}  // namespace
