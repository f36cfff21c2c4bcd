// Host-side runtime plumbing shared by the launchers: error reporting and launch checks.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/powerinfer_hip.h"

namespace pi {

// Weights that a launch requests ahead of the one that reads them (load_ahead in kernels_common.hpp): up to two matrices in units of unit_bytes (a
// multiple of 16), unit u by workgroups of XCD u % 8.  blocks: extra workgroups of the launch, a multiple of 8; 0: none.
struct Ahead { const void * p[2] = {nullptr, nullptr}; int units[2] = {0, 0}, unit_bytes[2] = {0, 0}, blocks = 0; };

void set_error(const char * msg);
int  fail(int code, const char * msg);                 // records msg, returns code
int  hip_fail(hipError_t e, const char * what);        // records "what: hipGetErrorString", returns PI_E_HIP
int  check_launch(const char * what);                  // hipGetLastError() after a kernel launch
int  compute_units();                                  // compute units of the current device (0 on error); cached per device, allocates nothing
int  noalloc_setup();                                  // resolves the static scratch array of pi_k_sparse_ffn_noalloc on the current device

// pi_k_attn_fused with such extra workgroups
int attn_fused(const float * qkv, const void * rope_table, void * k_cache, void * v_cache, int n_head, int n_head_kv, int hd, int mode,
               int n_ctx, const int32_t * pos, float * out, const Ahead & ahead, pi_stream_t stream);

}  // namespace pi

#define PI_HIP_TRY(expr)                                          \
    do {                                                          \
        hipError_t _e = (expr);                                   \
        if (_e != hipSuccess) return pi::hip_fail(_e, #expr);     \
    } while (0)
