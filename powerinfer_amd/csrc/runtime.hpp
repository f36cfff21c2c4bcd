// Host-side runtime plumbing shared by the launchers: error reporting and launch checks.
#pragma once

#include <hip/hip_runtime.h>

namespace pi {

void set_error(const char * msg);
int  fail(int code, const char * msg);                 // records msg, returns code
int  hip_fail(hipError_t e, const char * what);        // records "what: hipGetErrorString", returns PI_E_HIP
int  check_launch(const char * what);                  // hipGetLastError() after a kernel launch
int  compute_units();                                  // compute units of the current device (0 on error); cached per device, allocates nothing
// attention of a prompt chunk by 64 or 128 tokens of a head at a time (kernels_attn.hip): whether it covers a call, and the launches
bool attn_chunk_rows_fits(int hd, int T, int n_kv_max, const void * out, const void * out_f16, int out_stride);
int  attn_chunk_rows(const float * qkv, int qkv_stride, int T, int n_head, int n_head_kv, int hd, int mode, float theta_scale, float freq_scale, const int * pos, int n_ctx,
                     int n_kv_max, float * q_rot, void * k_cache, void * v_cache, float * out, int out_stride, void * out_f16, hipStream_t st);
int  noalloc_setup();                                  // resolves the static scratch array of pi_k_sparse_ffn_noalloc on the current device

}  // namespace pi

#define PI_HIP_TRY(expr)                                          \
    do {                                                          \
        hipError_t _e = (expr);                                   \
        if (_e != hipSuccess) return pi::hip_fail(_e, #expr);     \
    } while (0)
