// The HIP and hipBLASLt entry points this library calls, on the CPU: memory is host memory (counted, with a limit), a launch runs nothing, is
// counted by its kernel's name and fails on request.  Host code - what is allocated, which kernels a call takes, which errors it
// reports - runs unchanged on top.  Loaded with RTLD_GLOBAL in front of the library.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <hipblaslt/hipblaslt.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void *, std::string> & names() { static std::map<const void *, std::string> m; return m; }
std::map<std::string, int> counts;
std::map<void *, size_t> live;
size_t live_bytes = 0, peak_bytes = 0, limit_bytes = ~(size_t)0;
int n_launch = 0, fail_at = -1, grid_x = 0;
hipError_t last = hipSuccess;
void (*watcher)(const char *, void **) = nullptr;
char some[64];
template <typename T> hipError_t give(T * p) { *p = (T)some; return hipSuccess; }
}  // namespace

extern "C" {
void fake_fail_launch(int k) { n_launch = 0; fail_at = k; last = hipSuccess; }
int fake_launches() { return n_launch; }
void fake_watch(void (*f)(const char *, void **)) { watcher = f; }      // called with the name and the arguments of every launch that does not fail
int fake_grid() { return grid_x; }                     // workgroups of the last launch
void fake_limit(size_t free_bytes) { limit_bytes = free_bytes == ~(size_t)0 ? free_bytes : live_bytes + free_bytes; }
size_t fake_live() { return live_bytes; }
size_t fake_peak() { size_t p = peak_bytes; peak_bytes = live_bytes; return p; }
void fake_clear_counts() { counts.clear(); }
int fake_count(const char * part) {                    // launches since then of kernels whose name holds `part`
    int n = 0;
    for (auto & c : counts) if (c.first.find(part) != std::string::npos) n += c.second;
    return n;
}

void ** __hipRegisterFatBinary(const void *) { return (void **)some; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void * f, char *, const char * name, unsigned, void *, void *, void *, void *, int *) { names()[f] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3, size_t, hipStream_t) { grid_x = g.x; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 * g, dim3 * b, size_t * sh, hipStream_t * st) { *g = dim3(1); *b = dim3(1); *sh = 0; *st = nullptr; return hipSuccess; }
hipError_t hipLaunchKernel(const void * f, dim3, dim3, void ** args, size_t, hipStream_t) {
    ++counts[names()[f]];
    if (n_launch++ == fail_at) return last = hipErrorInvalidValue;
    if (watcher) watcher(names()[f].c_str(), args);
    return hipSuccess;
}
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
const char * hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int * v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevice(int * d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int * n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t * p, int) { memset(p, 0, sizeof *p); p->warpSize = 64; p->multiProcessorCount = 256; strcpy(p->gcnArchName, "gfx950"); return hipSuccess; }
hipError_t hipGetSymbolAddress(void ** p, const void *) { return give(p); }
hipError_t hipMemGetInfo(size_t * f, size_t * t) { *t = (size_t)288 << 30; *f = *t - live_bytes; return hipSuccess; }

hipError_t hipMalloc(void ** p, size_t n) {
    if (live_bytes + n > limit_bytes) { *p = nullptr; return last = hipErrorOutOfMemory; }
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    live[*p] = n; live_bytes += n;
    if (live_bytes > peak_bytes) peak_bytes = live_bytes;
    return hipSuccess;
}
hipError_t hipFree(void * p) {
    auto it = live.find(p);
    if (it == live.end()) return p ? hipErrorInvalidValue : hipSuccess;
    live_bytes -= it->second; live.erase(it); free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void ** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void * p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void * d, const void * s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void * d, const void * s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2DAsync(void * d, size_t dp, const void * s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    for (size_t i = 0; i < h; ++i) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemset(void * d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void * d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }

hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t * s, unsigned) { return give(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t * g) { return give(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t * e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return give(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t * e) { return give(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t * e, unsigned) { return give(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float * ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }

hipblasStatus_t hipblasLtCreate(hipblasLtHandle_t * h) { *h = some; return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtDestroy(const hipblasLtHandle_t) { return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulDescCreate(hipblasLtMatmulDesc_t * d, hipblasComputeType_t, hipDataType) { *d = (hipblasLtMatmulDesc_t)some; return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulDescDestroy(const hipblasLtMatmulDesc_t) { return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulDescSetAttribute(hipblasLtMatmulDesc_t, hipblasLtMatmulDescAttributes_t, const void *, size_t) { return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatrixLayoutCreate(hipblasLtMatrixLayout_t * l, hipDataType, uint64_t, uint64_t, int64_t) { *l = (hipblasLtMatrixLayout_t)some; return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatrixLayoutDestroy(const hipblasLtMatrixLayout_t) { return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulPreferenceCreate(hipblasLtMatmulPreference_t * p) { *p = (hipblasLtMatmulPreference_t)some; return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulPreferenceDestroy(const hipblasLtMatmulPreference_t) { return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulPreferenceSetAttribute(hipblasLtMatmulPreference_t, hipblasLtMatmulPreferenceAttributes_t, const void *, size_t) { return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmulAlgoGetHeuristic(hipblasLtHandle_t, hipblasLtMatmulDesc_t, hipblasLtMatrixLayout_t, hipblasLtMatrixLayout_t, hipblasLtMatrixLayout_t, hipblasLtMatrixLayout_t,
                                                hipblasLtMatmulPreference_t, const int, hipblasLtMatmulHeuristicResult_t r[], int * n) { r[0] = {}; *n = 1; return HIPBLAS_STATUS_SUCCESS; }
hipblasStatus_t hipblasLtMatmul(hipblasLtHandle_t, hipblasLtMatmulDesc_t, const void *, const void *, hipblasLtMatrixLayout_t, const void *, hipblasLtMatrixLayout_t, const void *, const void *,
                                hipblasLtMatrixLayout_t, void *, hipblasLtMatrixLayout_t, const hipblasLtMatmulAlgo_t *, void *, size_t, hipStream_t) {
    ++counts["hipblasLtMatmul"];
    return HIPBLAS_STATUS_SUCCESS;
}
}
