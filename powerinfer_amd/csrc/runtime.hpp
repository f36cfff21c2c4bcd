// Host-side runtime plumbing shared by the launchers: error reporting and launch checks.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/powerinfer_hip.h"

#include <stddef.h>

namespace pi {

// Weights that a launch requests ahead of the one that reads them (load_ahead in kernels_common.hpp): up to two matrices in units of unit_bytes (a
// multiple of 16), unit u by workgroups of XCD u % 8.  blocks: extra workgroups of the launch, a multiple of 8; 0: none.
struct Ahead { const void * p[2] = {nullptr, nullptr}; int units[2] = {0, 0}, unit_bytes[2] = {0, 0}, blocks = 0; };

void set_error(const char * msg);
int  fail(int code, const char * msg);                 // records msg, returns code
int  hip_fail(hipError_t e, const char * what);        // records "what: hipGetErrorString", returns PI_E_HIP
[[nodiscard]] int check_launch(const char * what);                  // hipGetLastError() after a kernel launch
int  compute_units();                                  // compute units of the current device (0 on error); cached per device, allocates nothing
int  noalloc_setup();                                  // resolves the static scratch array of pi_k_sparse_ffn_noalloc on the current device

// A call's results on their way from the device to the caller's memory.  A copy to pageable memory costs 13 us for 4 bytes and 62 us for the
// 128 KB of 32000 logits, each with a wait of its own; here one small kernel behind the call's last one stores all of them in pinned
// memory, one wait covers both, and a memcpy (3 us for 128 KB, still in the host's cache) brings them home.  Larger results (2 MB: 16
// rows of logits) travel in pieces of 512 KB, each copied while the next ones cross the link.  Part of one model, used by one call at a time.
// Pinning 2 MB takes 0.7 ms and the first call on them 0.2 to 0.3 ms more: a model that goes leaves its memory to the next ones (at most kKept
// such buffers; the last model of the process gives all of them back).
// A launch that stores results says so in words of the pinned memory, behind its stores, and the host looks there: the runtime's own wait puts a packet behind
// the launch, 5 us a token, and takes 30 us where the work has ended before it is called (the last piece of several).  Us, stream wait and events / this: 8 tokens of a 7B shape of 4
// layers 2254 -> 2201, of three layers of 512 x 4096 830 -> 780, of Falcon-40B's of 4 4641 -> 4582; 4 steps of 16 sequences (13B, 4 layers) 3252 -> 3200; a prompt pass and 12
// steps of 16 requests 17180 -> 16790; a prompt of 333 and 16 tokens 9220 -> 8950.  (Before the wait behind the write-back, pi_release, without which a word may get ahead of its
// values; with it these are as fast within the spread.)
struct HostDone { uint32_t * word; uint32_t value; };
struct HostAsk { uint32_t * word = nullptr; uint32_t tag = 0; };
struct HostCopy { const void * dev; void * host; size_t bytes; };        // multiples of 4 bytes, dev 4-byte aligned; host null: not wanted
struct HostStage {
    static constexpr int kPieces = 4, kMaxCopies = 4, kKept = 4, kBlocks = 64;      // (kBlocks: workgroups of a copy)
    static constexpr size_t kPiece = (size_t)512 << 10;
    unsigned char * pin = nullptr;         // null (no pinned memory to be had): ordinary copies
    size_t piece = 0; int n_pieces = 0;
    bool counted = false, busy = false;    // one of the pool's users; a call ended early, work on the memory may be left
    uint32_t * told = nullptr, asked = 0;  // a word behind those: what a launch in the middle of a call says, for what the host queues next, and the tag of the last question
    uint32_t * done = nullptr, seq = 0;    // [kPieces][kBlocks] behind the pieces: where the workgroups that store results say that they are through, and what the last launch's say
    void init(size_t usual_bytes);
    void release();
    // queues the copies behind what the stream holds and returns when the stream is done and the results are in place; all but the
    // last copy together fit in 4 KB of the first piece (else ordinary copies)
    int fetch(const HostCopy * copies, int n, hipStream_t st);
    // room for results that the call's own last launch stores (null: to be had with fetch only), and the wait for them
    unsigned char * room(size_t bytes) { if (!pin || bytes > piece) return nullptr; busy = true; return pin; }
    HostDone next(int slot = 0) { return {done + slot * kBlocks, ++seq}; }
    // for the launch that the last `next()` went to, the last of the stream, one of whose workgroups speaks for all; apart: the runtime's wait, which leaves the core to others
    int wait(hipStream_t st, bool apart = false);
    int until(const HostDone & d, int words, hipStream_t st);
    // a question that a launch to come answers with tag | a number of 16 bits (word null: nowhere to), and the wait for the answer, which may have much ahead of it: the host looks rarely
    // before long.  The tags differ, so that an answer left by a call that failed is nobody's.
    HostAsk ask() { asked += 1u << 16; if (!asked) asked = 1u << 16; return {told, asked}; }
    int answer(hipStream_t st, uint32_t * value);
};

// pi_k_attn_fused with such extra workgroups
int attn_fused(const float * qkv, const void * rope_table, void * k_cache, void * v_cache, int n_head, int n_head_kv, int hd, int mode,
               int n_ctx, const int32_t * pos, float * out, const Ahead & ahead, pi_stream_t stream);
// Attention of one decoded token and its sparse FFN's partial vectors in one launch (attn_ffn_kernel): what pi_k_attn_split (n_parts > 1: scratch) or pi_k_attn_fused and
// pi_k_sparse_ffn_partials leave
struct DecodeAttn { const float * qkv; const void * rope_table; void * k_cache, * v_cache; int n_head, n_head_kv, hd, mode, n_ctx, n_parts; const int32_t * pos; float * scratch, * out; uint32_t * arrived; };   // arrived: [n_head], 0 between two launches
// Attention and output projection of one decoded token of a small model in one launch: parts[h] [d], a head's share of wo att (attn_out_small_kernel)
constexpr int kOutHeads = 16;
bool attn_out_small_supported(int n_head, int hd, int n_ctx);
int attn_out_small(const DecodeAttn & a, const void * wo_f16, int d, float * parts, pi_stream_t stream);
// pi_k_sparse_ffn_small of x + the n_parts vectors of `parts`, which go to xsum as well and are its residual
int sparse_ffn_small_of(const float * parts, int n_parts, float * xsum, const void * fc1_f16, const void * fc2_f16, int ff, int r, float threshold, const void * up_f16, const void * gate_f16,
                        const void * down_t_f16, int cols, const float * x, const pi_norm * norm, float * out, int32_t * n_active, pi_workspace * ws, pi_stream_t stream);
bool attn_ffn_supported(const void * fc2_f16, int ff, int r, int cols, int hd, int n_ctx, int n_parts);
int attn_ffn(const DecodeAttn & a, const void * fc2_f16, int ff, int r, const float * hidden, float threshold, const void * up_f16, const void * down_t_f16, int cols, const float * x, const pi_norm * norm,
             pi_workspace * ws, pi_stream_t stream);
// two mat-vecs of one vector in one launch (F16, 8192 columns): y = W norm(x), LayerNorm with its bias, and y2 = relu(W2 x)
bool gemv_pair_supported(int type, int type2, int cols, const pi_norm * norm, const float * x);
// y = W x + resid + the vectors of the workspace's sparse FFN (F16, 8192 columns and rows), and its active neurons
int gemv_ffn_out(const void * W, int cols, const float * x, const float * resid, float * y, int32_t * n_active, pi_workspace * ws, pi_stream_t stream);
int gemv_pair(const void * W, int rows, const pi_norm * norm, float * y, const void * W2, int rows2, float * y2, int cols, const float * x, pi_stream_t stream);
// What a pass of a model of layers begins with (pass_start_kernel): words from src to dst; triples (sequence, place, cell) into lists; T embeddings (table null:
// none) with a norm or a scale and bigrams; angles of up to kRots rotations (freq null: from base).
struct PassStart {
    static constexpr int kRots = 8;
    struct Rot { int dims; double base, length; const double * freq; void * cs; };
    const int32_t * src; int32_t * dst; size_t words;
    const int32_t * append; int n_append; int32_t * lists; size_t list_ld;
    const void * table; int cols, T; const int32_t * tokens, * prev, * pos; const float * norm; float eps, scale;
    const void * bigram; int buckets; int64_t mul_prev, mul_cur; float * x, * x0;
    int n_rot; Rot rot[kRots];
};
int pass_start(const PassStart & p, hipStream_t st);
// whether pi_k_attn_chunk takes the tokens of a chunk against n_kv_max cells 16 at a time on the matrix cores
bool attn_chunk_by_16(int hd, int n_kv_max);
int rope_kv_chunk(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale, const int32_t * pos, int n_ctx,
                  float * q_rot, void * k_cache, void * v_cache, hipStream_t st, bool q16 = false);
// pi_k_expert_up_step with act = weight * relu(up[e] x)^2 (up [n_expert][ff][cols])
int expert_relu2_step(const void * up, int n_expert, int ff, int cols, const void * x_ol, int T, const int32_t * ids, const float * weights, int top, void * act, int ld_act,
                      pi_stream_t stream);
// the embedding row of a token that the host names; also writes the token loop's state (token, position, step counter 0)
int embed_start(int wtype, const void * table, int cols, int32_t token, int32_t pos, int32_t * d_token, int32_t * d_pos, int32_t * d_step, float * x, pi_stream_t stream);
// where a prompt's last token goes on alone behind a chunk that it came along in: its input of the next layer, and the loop's state as embed_start leaves it
int resume_token(const float * row, int cols, int32_t token, int32_t pos, int32_t * d_token, int32_t * d_pos, int32_t * d_step, float * x, pi_stream_t stream);
// how many neurons of a chunk's last token (T of them) fire, by the predictor's logits [T][ff] or its bits (pi_k_ffn_wide_predicted_f16)
int count_active(const float * logits, const void * mask, int T, int ff, float thr, int32_t * n_active, pi_stream_t stream);
// the predictor's bits of a chunk (pi_k_ffn_wide_predicted_f16, which checks the operands) and, where `any` is not null, 64 tokens at a time, which neurons fire for one of them, a bit a neuron
int predictor_bits(const void * fc2_f16, int ff, int rank, const void * hid_f16, int T, float threshold, void * mask, void * any, pi_stream_t stream);
// The two halves of pi_k_ffn_union_f16, checked as there: predictor bits, list and h [T][number of listed ones], which `told` gets too (ff: all of them, and in their order), and the down projection
int ffn_union_hidden(const void * fc2_f16, int rank, const void * hid_f16, const void * up_f16, const void * gate_f16, int ff, int cols, const void * xn_f16, int T, float threshold, void * scratch,
                     void * h_f16, int32_t * n_active, const HostAsk & told, pi_stream_t stream);
int ffn_union_down(const void * down_t_f16, int ff, int cols, int T, const void * scratch, const void * h_f16, float * const * parts, const float * add1, const float * add2, float * out, pi_stream_t stream);
// the embedding rows of tokens that the host names, at positions from `pos` on, and these positions
int embed_chunk(int wtype, const void * table, int cols, const int32_t * tokens, int T, int pos, float * x, int32_t * d_pos, pi_stream_t stream);

}  // namespace pi

#define PI_HIP_TRY(expr)                                          \
    do {                                                          \
        hipError_t _e = (expr);                                   \
        if (_e != hipSuccess) return pi::hip_fail(_e, #expr);     \
    } while (0)
