// The host-pointer form without a GPU: the host code of host_call.hip with stand-ins for the HIP calls it makes.
// Allocation number n of a call fails, for every n until a call gets through: whatever the point of failure, nothing may
// be left on the streams, whose copies read and write the pinned pieces that the next call uses.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <hip/hip_runtime.h>
#include "../sddmm_gpu_amd/csrc/host_call.hip"

static std::atomic<int> allocations_left{-1};  // (negative: none fails)
void *operator new(size_t n)
{
    if (allocations_left.load() >= 0 && allocations_left.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void *p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

static std::mutex mu;
static int busy_streams[8];  // work put on a stream and not waited for
static int n_streams = 0, device_arrays = 0;
static void work(hipStream_t s) { std::lock_guard<std::mutex> g(mu); busy_streams[(intptr_t)s & 7] = 1; }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n); ++device_arrays; return hipSuccess; }
hipError_t hipFree(void *p) { free(p); --device_arrays; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)(intptr_t)(1 + n_streams++ % 7); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { std::lock_guard<std::mutex> g(mu); busy_streams[(intptr_t)s & 7] = 0; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s) { work(s); return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s);
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s);
static thread_local hipStream_t pushed;
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s) { pushed = s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) { *g = dim3(1); *b = dim3(1); *n = 0; *s = pushed; return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *p; return &p; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, dim3 *, dim3 *, int *) {}
extern const char __hip_fatbin[] __attribute__((weak)) = "";
int sddmm_execute(const sddmm_plan *, const float *, const float *, const float *, float *, void *stream) { work((hipStream_t)stream); return SDDMM_OK; }
}
namespace sddmm {
int fail(int code, const char *, ...) { return code; }
}

int main()
{
    int failed = 0;
    for (int n = 0;; ++n) {
        sddmm_plan plan;
        plan.info.n_rows = 3 << 18; plan.info.n_cols = 1 << 10; plan.info.K = 4; plan.info.nnz = 5 << 20;
        std::vector<float> W((size_t)plan.info.n_rows * 4), H((size_t)plan.info.n_cols * 4), out((size_t)plan.info.nnz);
        allocations_left = n;
        const int rc = sddmm_gpu(&plan, W.data(), H.data(), out.data(), nullptr);
        const bool through = allocations_left.load() >= 0;
        allocations_left = -1;
        if (rc != SDDMM_OK) {
            ++failed;
            for (int s = 0; s < 8; ++s)
                if (busy_streams[s]) { printf("allocation %d failed (code %d): work left on stream %d\n", n, rc, s); return 1; }
        }
        memset(busy_streams, 0, sizeof busy_streams);
        if (through) break;
        if (n > 1000) return 2;
    }
    if (device_arrays) { printf("%d device arrays not freed\n", device_arrays); return 3; }
    printf("%d points of failure\n", failed);
    return failed >= 5 ? 0 : 4;
}
