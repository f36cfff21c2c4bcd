// Device/runtime plumbing of the C ABI: init, memory, copies, events, error string.
#include <chrono>
#include <mutex>
#include <thread>
#include "device_utils.hpp"
#include "runtime.hpp"
#include "../../include/powerinfer_hip.h"

#include <stdio.h>
#include <string.h>

namespace pi {

static thread_local char g_err[512] = "";

void set_error(const char * msg) { snprintf(g_err, sizeof g_err, "%s", msg); }
int fail(int code, const char * msg) { set_error(msg); return code; }
int hip_fail(hipError_t e, const char * what) {
    snprintf(g_err, sizeof g_err, "%s: %s", what, hipGetErrorString(e));
    return PI_E_HIP;
}
int check_launch(const char * what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PI_OK : hip_fail(e, what);
}

}  // namespace pi

namespace pi {
int compute_units() {
    static int cached[16] = {};
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 0;
    if (!cached[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
        cached[dev] = n;
    }
    return cached[dev];
}
}  // namespace pi

namespace {
struct CopyOut { const uint32_t * src[pi::HostStage::kMaxCopies]; uint32_t words[pi::HostStage::kMaxCopies], at[pi::HostStage::kMaxCopies]; };
__global__ __launch_bounds__(256) void copy_out_kernel(CopyOut c, uint32_t * __restrict__ dst, pi::HostDone done) {
    const uint32_t i0 = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
#pragma unroll
    for (int r = 0; r < pi::HostStage::kMaxCopies; ++r) {
        const uint32_t * s = c.src[r];
        uint32_t * d = dst + c.at[r];
        uint32_t done4 = 0;
        if (((uintptr_t)s & 15) == 0) {                             // (places in the buffer are multiples of 64 bytes)
            const uint32_t n4 = c.words[r] / 4;
            for (uint32_t i = i0; i < n4; i += step) reinterpret_cast<uint4 *>(d)[i] = reinterpret_cast<const uint4 *>(s)[i];
            done4 = n4 * 4;
        }
        for (uint32_t i = done4 + i0; i < c.words[r]; i += step) d[i] = s[i];
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                             // vmcnt(0): this wave's stores are under way
    __syncthreads();
    if (threadIdx.x == 0) {
        pi_release<true>();
        __hip_atomic_store(done.word + blockIdx.x, done.value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
}  // namespace

namespace pi {
namespace {
std::mutex pinned_lock;
struct { unsigned char * p; size_t bytes; } pinned_kept[HostStage::kKept];
int pinned_n = 0, pinned_users = 0;
}  // namespace

void HostStage::init(size_t usual_bytes) {
    if (counted) return;
    const size_t want = usual_bytes + 4096;
    n_pieces = want > kPiece ? kPieces : 1;
    piece = n_pieces > 1 ? kPiece : (want + 4095) / 4096 * 4096;
    counted = true;
    {
        std::lock_guard<std::mutex> held(pinned_lock);
        ++pinned_users;
        for (int i = 0; i < pinned_n && !pin; ++i)
            if (pinned_kept[i].bytes == piece * n_pieces) { pin = pinned_kept[i].p; pinned_kept[i] = pinned_kept[--pinned_n]; }
    }
    if (!pin && hipHostMalloc((void **)&pin, piece * n_pieces + 4 * kPieces * kBlocks + 64, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) { pin = nullptr; (void)hipGetLastError(); return; }
    done = reinterpret_cast<uint32_t *>(pin + piece * n_pieces);
    told = done + kPieces * kBlocks;
    memset(done, 0, 4 * kPieces * kBlocks + 64);
    seq = asked = 0;
}

void HostStage::release() {
    if (!counted) return;
    counted = false;
    unsigned char * out[kKept + 1];
    int n = 0;
    {
        std::lock_guard<std::mutex> held(pinned_lock);
        if (pin && !busy && pinned_n < kKept) { pinned_kept[pinned_n].p = pin; pinned_kept[pinned_n++].bytes = piece * n_pieces; }
        else if (pin) out[n++] = pin;
        if (--pinned_users == 0) while (pinned_n) out[n++] = pinned_kept[--pinned_n].p;
    }
    pin = nullptr;
    told = nullptr;
    while (n) (void)hipHostFree(out[--n]);
}

int HostStage::until(const HostDone & d, int words, hipStream_t st) {
    const auto end = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
    for (int w = 0, k = 1; w < words; ++k) {
        if (__atomic_load_n(d.word + w, __ATOMIC_ACQUIRE) == d.value) { ++w; continue; }
        // what does not get through, or takes longer than a token, is the runtime's to wait for
        if (k % 64 == 0 && std::chrono::steady_clock::now() > end) { PI_HIP_TRY(hipStreamSynchronize(st)); return PI_OK; }
        __builtin_ia32_pause();
    }
    return PI_OK;
}
int HostStage::answer(hipStream_t st, uint32_t * value) {
    const auto soon = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
    const auto here = [&] {
        const uint32_t v = __atomic_load_n(told, __ATOMIC_ACQUIRE);
        *value = v & 0xFFFF;
        return (v & ~0xFFFFu) == asked;
    };
    for (int k = 1; !here(); ++k) {
        if (k % 64 || std::chrono::steady_clock::now() < soon) { __builtin_ia32_pause(); continue; }
        std::this_thread::sleep_for(std::chrono::microseconds(50));
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) { (void)hipGetLastError(); continue; }
        if (e != hipSuccess) return hip_fail(e, "HostStage::answer");
        if (!here()) return fail(PI_E_STATE, "HostStage::answer: no launch has answered");
        break;
    }
    return PI_OK;
}
int HostStage::wait(hipStream_t st, bool apart) {
    if (apart) PI_HIP_TRY(hipStreamSynchronize(st));
    else if (const int rc = until({done, seq}, 1, st)) return rc;
    busy = false;
    return PI_OK;
}

int HostStage::fetch(const HostCopy * copies, int n, hipStream_t st) {
    HostCopy c[kMaxCopies];
    int m = 0;
    size_t small = 0, at[kMaxCopies] = {};
    for (int i = 0; i < n; ++i)
        if (copies[i].host && copies[i].bytes) { if (m == kMaxCopies) return fail(PI_E_ARG, "fetch: too many results"); c[m++] = copies[i]; }
    for (int i = 0; i + 1 < m; ++i) { at[i] = small; small += (c[i].bytes + 63) / 64 * 64; }
    if (!pin || small > 4096) {
        PI_HIP_TRY(hipStreamSynchronize(st));
        for (int i = 0; i < m; ++i) PI_HIP_TRY(hipMemcpy(c[i].host, c[i].dev, c[i].bytes, hipMemcpyDeviceToHost));
        return PI_OK;
    }
    if (m == 0) { PI_HIP_TRY(hipStreamSynchronize(st)); return PI_OK; }
    busy = true;                                                    // until the stream has been waited for
    // the last result in pieces; the first one leaves room for the others
    const HostCopy & big = c[m - 1];
    size_t sent = 0, taken = 0;                                     // bytes of it
    size_t from[kPieces] = {}, len[kPieces] = {};
    HostDone through[kPieces] = {};
    int blocks[kPieces] = {};
    int queued = 0, fetched = 0;
    while (taken < big.bytes) {
        while (sent < big.bytes && queued - fetched < n_pieces) {
            const int slot = queued % n_pieces;
            const size_t head = queued ? 0 : small;
            const size_t b = big.bytes - sent < piece - head ? big.bytes - sent : piece - head;
            CopyOut o{};
            for (int i = 0; i + 1 < m && !queued; ++i) { o.src[i] = (const uint32_t *)c[i].dev; o.words[i] = (uint32_t)(c[i].bytes / 4); o.at[i] = (uint32_t)(at[i] / 4); }
            o.src[kMaxCopies - 1] = (const uint32_t *)((const unsigned char *)big.dev + sent); o.words[kMaxCopies - 1] = (uint32_t)(b / 4); o.at[kMaxCopies - 1] = (uint32_t)(head / 4);
            blocks[slot] = std::min(std::max((int)((b / 16 + 255) / 256), 1), kBlocks);
            through[slot] = next(slot);
            hipLaunchKernelGGL(copy_out_kernel, dim3(blocks[slot]), dim3(256), 0, st, o, reinterpret_cast<uint32_t *>(pin + (size_t)slot * piece), through[slot]);
            if (const int rc = check_launch("copy_out")) return rc;
            from[slot] = sent; len[slot] = b; sent += b; ++queued;
        }
        const int slot = fetched % n_pieces;
        if (const int rc = until(through[slot], blocks[slot], st)) return rc;      // (the last one: everything the stream held)
        const unsigned char * s = pin + (size_t)slot * piece;
        if (!fetched) for (int i = 0; i + 1 < m; ++i) memcpy(c[i].host, s + at[i], c[i].bytes);
        memcpy((unsigned char *)big.host + from[slot], s + (fetched ? 0 : small), len[slot]);
        taken += len[slot]; ++fetched;
    }
    busy = false;
    return PI_OK;
}
}  // namespace pi

extern "C" {

const char * pi_last_error(void) { return pi::g_err; }

int pi_init(int device) {
    int n = 0;
    PI_HIP_TRY(hipGetDeviceCount(&n));
    if (n <= 0) return pi::fail(PI_E_HIP, "pi_init: no HIP device; this library has no CPU fallback");
    if (device < 0 || device >= n) return pi::fail(PI_E_ARG, "pi_init: device index out of range");
    PI_HIP_TRY(hipSetDevice(device));
    hipDeviceProp_t p;
    PI_HIP_TRY(hipGetDeviceProperties(&p, device));
    if (p.warpSize != 64) return pi::fail(PI_E_UNSUPPORTED, "pi_init: kernels are written for 64-wide wavefronts");
    (void)pi::compute_units();
    return pi::noalloc_setup();
}

int pi_device_name(char * buf, size_t n) {
    int dev = 0;
    PI_HIP_TRY(hipGetDevice(&dev));
    hipDeviceProp_t p;
    PI_HIP_TRY(hipGetDeviceProperties(&p, dev));
    snprintf(buf, n, "%s (%s, %d CUs)", p.name, p.gcnArchName, p.multiProcessorCount);
    return PI_OK;
}

void * pi_malloc(size_t bytes) {
    void * p = nullptr;
    const hipError_t e = hipMalloc(&p, bytes ? bytes : 1);
    if (e != hipSuccess) { pi::hip_fail(e, "hipMalloc"); return nullptr; }
    return p;
}
int pi_free(void * dptr) { if (dptr) PI_HIP_TRY(hipFree(dptr)); return PI_OK; }
void * pi_malloc_host(size_t bytes) {
    void * p = nullptr;
    const hipError_t e = hipHostMalloc(&p, bytes ? bytes : 1, hipHostMallocCoherent);
    if (e != hipSuccess) { pi::hip_fail(e, "hipHostMalloc"); return nullptr; }
    return p;
}
int pi_free_host(void * hptr) { if (hptr) PI_HIP_TRY(hipHostFree(hptr)); return PI_OK; }
int pi_memset(void * dptr, int byte, size_t bytes) { PI_HIP_TRY(hipMemset(dptr, byte, bytes)); return PI_OK; }
int pi_memcpy_h2d(void * dptr, const void * host, size_t bytes) { PI_HIP_TRY(hipMemcpy(dptr, host, bytes, hipMemcpyHostToDevice)); return PI_OK; }
int pi_memcpy_d2h(void * host, const void * dptr, size_t bytes) { PI_HIP_TRY(hipMemcpy(host, dptr, bytes, hipMemcpyDeviceToHost)); return PI_OK; }
int pi_memcpy_d2d(void * dst, const void * src, size_t bytes) { PI_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice)); return PI_OK; }
int pi_sync(void) { PI_HIP_TRY(hipDeviceSynchronize()); return PI_OK; }

void * pi_event_create(void) {
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) { pi::set_error("hipEventCreate failed"); return nullptr; }
    return (void *)e;
}
int pi_event_record(void * ev, pi_stream_t stream) { PI_HIP_TRY(hipEventRecord((hipEvent_t)ev, (hipStream_t)stream)); return PI_OK; }
int pi_event_elapsed_ms(void * start, void * stop, float * ms) {
    PI_HIP_TRY(hipEventSynchronize((hipEvent_t)stop));
    PI_HIP_TRY(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
    return PI_OK;
}
int pi_event_destroy(void * ev) { PI_HIP_TRY(hipEventDestroy((hipEvent_t)ev)); return PI_OK; }

}  // extern "C"
