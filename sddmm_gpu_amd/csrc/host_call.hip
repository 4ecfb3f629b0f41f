// sddmm_gpu, the host-pointer form: W and H from host memory to the device, the plan's kernels, the results back.
//
// What bounds it is the host link (57 GB/s each way here).  The runtime's own copies of pageable memory reach 39
// GB/s up and 18 down on one thread, which also takes the page faults of a fresh output array one after the other,
// so the copies go through pinned pieces here: a few threads copy between the caller's memory and the pieces while
// a copy kernel per piece moves the ones before over the link, on three streams so that one kernel's start hides
// behind another's work.  27.4 MB up and 19.5 MB down: 2.20 -> 1.13 ms a call (0.83 ms of it the link).  The pieces, streams and
// threads (HostPipe) are shared by all plans that have made such a call and go with the last of them; the device
// arrays stay with their plan, until it is destroyed or sddmm_plan_release_host.
#include <hip/hip_runtime.h>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include "plan.hpp"

using namespace sddmm;

namespace {

typedef float vec4f __attribute__((ext_vector_type(4)));

// n4 pieces of 16 bytes and `tail` floats, to or from pinned host memory (16-byte aligned).  16 workgroups with
// four requests per thread, on three streams, keep more than the link's bandwidth times its latency in flight, and one
// kernel's start and end hide behind two others (27.4 MB up, 19.5 MB down, us a call: 32 workgroups on one / two / four streams
// 1416 / 1208 / 1203, 16 on two / three / four 1176 / 1131 / 1162, 8 on two / four 1167 / 1135, 64 on two 1295).
constexpr int kCopyBlocks = 16;
__global__ __launch_bounds__(256)
void sddmm_host_copy_kernel(const vec4f *__restrict__ src, vec4f *__restrict__ dst, int n4, int tail)
{
    constexpr int stride = kCopyBlocks * 256;
    int i = blockIdx.x * 256 + threadIdx.x;
    for (; i + 3 * stride < n4; i += 4 * stride) {
        vec4f v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = __builtin_nontemporal_load(src + i + u * stride);
#pragma unroll
        for (int u = 0; u < 4; ++u) __builtin_nontemporal_store(v[u], dst + i + u * stride);
    }
    for (; i < n4; i += stride) dst[i] = src[i];
    if (blockIdx.x == 0 && (int)threadIdx.x < tail)
        reinterpret_cast<float *>(dst + n4)[threadIdx.x] = reinterpret_cast<const float *>(src + n4)[threadIdx.x];
}

}  // namespace

namespace sddmm {

// Pinned pieces, the threads that fill and empty them and the streams that move them, for one device.
class HostPipe {
public:
    static constexpr size_t kPiece = (size_t)1 << 20;
    static constexpr int kThreads = 8;            // the caller and seven more
    static constexpr int kPieces = 2 * kThreads;  // a thread works on one of its pieces while the other is on its way
    static constexpr int kStreams = 3;

    hipStream_t stream[kStreams] = {};  // (a thread's pieces all travel on one of them)
    hipEvent_t fork = nullptr, join[kStreams] = {}, e0 = nullptr, e1 = nullptr;
    std::mutex busy;  // held by a call from its first piece to its last
    // Streams of the call that holds it: small calls wait for more events than the streams hide.  us a call, one / two / three: 0.9 MB
    // 112 / 123 / 134, 1.3 MB 126 / 134 / 139, 2.4 MB 186 / 175 / 180, 3.5 MB 225 / 204 / 208, 5.2 MB 290 / 254 / 247, 14.7 MB 581 / 487 / 472.
    int used = kStreams;

    // the pipe of `device` (the current one), made if no plan holds it
    static std::shared_ptr<HostPipe> get(int device)
    {
        constexpr int kMaxDevices = 64;
        static std::mutex mu;
        static std::weak_ptr<HostPipe> held[kMaxDevices];
        if (device < 0 || device >= kMaxDevices) return nullptr;
        std::lock_guard<std::mutex> g(mu);
        if (auto p = held[device].lock()) return p;
        std::shared_ptr<HostPipe> p(new HostPipe);
        p->device = device;
        bool ok = hipHostMalloc((void **)&p->pinned, kPieces * kPiece, hipHostMallocDefault) == hipSuccess;
        for (auto &s : p->stream) ok = ok && hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess;
        for (auto &e : p->piece_done) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        for (auto &e : p->join) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        ok = ok && hipEventCreateWithFlags(&p->fork, hipEventDisableTiming) == hipSuccess;
        ok = ok && hipEventCreate(&p->e0) == hipSuccess && hipEventCreate(&p->e1) == hipSuccess;
        if (!ok) return nullptr;
        held[device] = p;
        return p;
    }

    ~HostPipe()
    {
        {
            std::lock_guard<std::mutex> g(mu);
            stop = true;
        }
        wake.notify_all();
        for (auto &t : threads) t.join();
        for (hipEvent_t e : piece_done) if (e) (void)hipEventDestroy(e);
        for (hipEvent_t e : join) if (e) (void)hipEventDestroy(e);
        for (hipEvent_t e : {fork, e0, e1}) if (e) (void)hipEventDestroy(e);
        for (hipStream_t s : stream) if (s) (void)hipStreamDestroy(s);
        if (pinned) (void)hipHostFree(pinned);
    }

    struct Part {
        const char *src;
        char *dst;
        size_t bytes;
    };

    // Host to device (up) or back, all parts.  Up: returns when the caller's memory has been read and every copy is
    // on the streams; down: when the caller's memory is written.  (The caller holds `busy` from before the way up to
    // after the way down, and the way down is ordered behind the way up on the device, so a piece is free again by then.)
    hipError_t move(const Part *parts, int n_parts, bool up)
    {
        Job j;
        j.up = up;
        // Pieces of 1 MB; while the first ones are filled (up) or the last ones emptied (down) the link is idle, so
        // every thread begins (ends) with a quarter and a half of one.
        size_t total = 0;
        for (int i = 0; i < n_parts; ++i) total += parts[i].bytes;
        size_t done = 0;
        for (int i = 0; i < n_parts; ++i)
            for (size_t o = 0; o < parts[i].bytes;) {
                const size_t edge = up ? done : total - done;
                size_t n = edge < kThreads * (kPiece / 4) ? kPiece / 4 : edge < kThreads * 3 * (kPiece / 4) ? kPiece / 2 : kPiece;
                n = std::min(n, parts[i].bytes - o);
                j.pieces.push_back({parts[i].src + o, parts[i].dst + o, n});
                o += n;
                done += n;
            }
        if (j.pieces.empty()) return hipSuccess;
        const int want = (int)std::min<size_t>(kThreads, j.pieces.size()) - 1;
        {
            std::lock_guard<std::mutex> g(mu);
            try {
                while ((int)threads.size() < want) {
                    const int id = (int)threads.size() + 1;
                    threads.emplace_back([this, id] { worker(id); });
                }
            } catch (const std::system_error &) {  // (no more threads to be had: the others do the work)
            }
            job = &j;
            wanted = pending = std::min<int>(want, (int)threads.size());
            ++generation;
        }
        wake.notify_all();
        run(j, 0);
        std::unique_lock<std::mutex> lk(mu);
        finished.wait(lk, [&] { return pending == 0; });
        job = nullptr;
        return j.err.load();
    }

private:
    struct Job {
        bool up = false;
        std::vector<Part> pieces;
        std::atomic<size_t> next{0};
        std::atomic<hipError_t> err{hipSuccess};
    };

    int device = 0;
    char *pinned = nullptr;
    hipEvent_t piece_done[kPieces] = {};
    std::vector<std::thread> threads;
    std::mutex mu;
    std::condition_variable wake, finished;
    Job *job = nullptr;
    uint64_t generation = 0;
    int wanted = 0, pending = 0;
    bool stop = false;

    void worker(int id)
    {
        uint64_t seen = 0;
        for (;;) {
            Job *j = nullptr;
            {
                std::unique_lock<std::mutex> lk(mu);
                wake.wait(lk, [&] { return stop || generation != seen; });
                if (stop) return;
                seen = generation;
                if (id > wanted || !job) continue;
                j = job;
            }
            run(*j, id);
            std::lock_guard<std::mutex> g(mu);
            if (--pending == 0) finished.notify_one();
        }
    }

    // Thread `id` takes pieces of the job one by one, through its own two pinned pieces.
    void run(Job &j, int id)
    {
        auto check = [&](hipError_t e) {
            if (e != hipSuccess) {
                hipError_t none = hipSuccess;
                j.err.compare_exchange_strong(none, e);
                j.next.store(j.pieces.size());  // the others stop at their next piece
            }
            return e == hipSuccess;
        };
        if (id > 0 && !check(hipSetDevice(device))) return;
        const hipStream_t st = stream[id % used];
        const Part *slot[2] = {};  // what travels through each of the two
        auto finish = [&](int k) {  // waits for the slot's copy; down: hands its bytes on
            const Part *p = slot[k];
            if (!p) return true;
            slot[k] = nullptr;
            if (!check(hipEventSynchronize(piece_done[2 * id + k]))) return false;
            if (!j.up) memcpy(p->dst, pinned + (2 * id + k) * kPiece, p->bytes);
            return true;
        };
        int k = 0;
        for (;; k ^= 1) {
            const size_t at = j.next.fetch_add(1);
            if (at >= j.pieces.size()) break;
            const Part &p = j.pieces[at];
            if (!finish(k)) return;
            char *pin = pinned + (2 * id + k) * kPiece;
            if (j.up) memcpy(pin, p.src, p.bytes);
            const int n4 = (int)(p.bytes / 16), tail = (int)(p.bytes % 16 / 4);
            hipLaunchKernelGGL(sddmm_host_copy_kernel, dim3(kCopyBlocks), dim3(256), 0, st, reinterpret_cast<const vec4f *>(j.up ? pin : p.src),
                               reinterpret_cast<vec4f *>(j.up ? p.dst : pin), n4, tail);
            if (!check(hipGetLastError()) || !check(hipEventRecord(piece_done[2 * id + k], st))) return;
            slot[k] = &p;
        }
        if (j.up) return;
        if (finish(k)) finish(k ^ 1);  // the older of the two first
    }
};

// What a plan keeps for its host calls.
struct HostCall {
    std::shared_ptr<HostPipe> pipe;
    int device = 0;
    float *W = nullptr, *H = nullptr, *out = nullptr;
    ~HostCall()
    {
        for (float *p : {W, H, out}) if (p) (void)hipFree(p);
    }
};

void HostCallDelete::operator()(HostCall *c) const { delete c; }

}  // namespace sddmm

namespace {

int make_host_call(const sddmm_plan *plan)
{
    const sddmm_plan_info &I = plan->info;
    std::unique_ptr<HostCall, HostCallDelete> c(new (std::nothrow) HostCall);
    if (!c) return fail(SDDMM_ERR_NOMEM, "sddmm_gpu: out of memory");
    HIP_TRY(hipGetDevice(&c->device));
    c->pipe = HostPipe::get(c->device);
    if (!c->pipe) return fail(SDDMM_ERR_HIP, "sddmm_gpu: cannot set up the host transfers: %s", hipGetErrorString(hipGetLastError()));
    const int64_t n[3] = {std::max<int64_t>(I.n_rows * (int64_t)I.K, 1), std::max<int64_t>(I.n_cols * (int64_t)I.K, 1), std::max<int64_t>(I.nnz, 1)};
    HIP_TRY(hipMalloc((void **)&c->W, (size_t)n[0] * 4));
    HIP_TRY(hipMalloc((void **)&c->H, (size_t)n[1] * 4));
    HIP_TRY(hipMalloc((void **)&c->out, (size_t)n[2] * 4));
    plan->host_call = std::move(c);
    plan->host_bytes = 4 * (n[0] + n[1] + n[2]);
    return SDDMM_OK;
}

int host_call(const sddmm_plan *plan, HostCall &c, const float *h_W, const float *h_H, float *h_out, float *kernel_ms)
{
    const sddmm_plan_info &I = plan->info;
    HostPipe &pipe = *c.pipe;
    // after whatever the caller has put on the default stream before
    HIP_TRY(hipEventRecord(pipe.fork, nullptr));
    const int64_t bytes = 4 * (I.n_rows * (int64_t)I.K + I.n_cols * (int64_t)I.K + I.nnz);
    pipe.used = bytes < ((int64_t)2 << 20) ? 1 : bytes < ((int64_t)4 << 20) ? 2 : HostPipe::kStreams;
    for (int i = 0; i < pipe.used; ++i) HIP_TRY(hipStreamWaitEvent(pipe.stream[i], pipe.fork, 0));
    const HostPipe::Part in[2] = {{(const char *)h_W, (char *)c.W, (size_t)I.n_rows * I.K * 4}, {(const char *)h_H, (char *)c.H, (size_t)I.n_cols * I.K * 4}};
    HIP_TRY(pipe.move(in, 2, true));
    for (int i = 1; i < pipe.used; ++i) {
        HIP_TRY(hipEventRecord(pipe.join[i], pipe.stream[i]));
        HIP_TRY(hipStreamWaitEvent(pipe.stream[0], pipe.join[i], 0));
    }
    HIP_TRY(hipEventRecord(pipe.e0, pipe.stream[0]));
    if (int rc = sddmm_execute(plan, nullptr, c.W, c.H, c.out, pipe.stream[0])) return rc;
    HIP_TRY(hipEventRecord(pipe.e1, pipe.stream[0]));
    for (int i = 1; i < pipe.used; ++i) HIP_TRY(hipStreamWaitEvent(pipe.stream[i], pipe.e1, 0));
    const HostPipe::Part back[1] = {{(const char *)c.out, (char *)h_out, (size_t)I.nnz * 4}};
    HIP_TRY(pipe.move(back, 1, false));
    HIP_TRY(hipEventSynchronize(pipe.e1));  // (there is nothing to copy back from an empty matrix)
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, pipe.e0, pipe.e1));
    if (kernel_ms) *kernel_ms = ms;
    return SDDMM_OK;
}

}  // namespace

extern "C" int sddmm_gpu(const sddmm_plan *plan, const float *h_W, const float *h_H, float *h_out, float *kernel_ms)
{
    if (!plan || !h_W || !h_H || !h_out) return fail(SDDMM_ERR_ARG, "sddmm_gpu: NULL argument");
    std::lock_guard<std::mutex> one(plan->host_mu);
    try {
        if (!plan->host_call)
            if (int rc = make_host_call(plan)) return rc;
        HostCall &c = *plan->host_call;
        int device = 0;
        HIP_TRY(hipGetDevice(&device));
        if (device != c.device) return fail(SDDMM_ERR_ARG, "sddmm_gpu: the plan's host calls belong to device %d, the current device is %d", c.device, device);
        std::lock_guard<std::mutex> transfer(c.pipe->busy);
        // nothing of a call that failed, by its code or by an exception, is left on the streams for the next one to meet
        struct Drain {
            HostPipe &pipe;
            bool failed = true;
            ~Drain()
            {
                if (failed)
                    for (hipStream_t s : pipe.stream) (void)hipStreamSynchronize(s);
            }
        } drain{*c.pipe};
        const int rc = host_call(plan, c, h_W, h_H, h_out, kernel_ms);
        drain.failed = rc != SDDMM_OK;
        return rc;
    } catch (const std::exception &e) {
        return fail(SDDMM_ERR_NOMEM, "sddmm_gpu: %s", e.what());
    }
}

extern "C" int sddmm_plan_release_host(const sddmm_plan *plan)
{
    if (!plan) return fail(SDDMM_ERR_ARG, "sddmm_plan_release_host: plan is NULL");
    std::lock_guard<std::mutex> one(plan->host_mu);
    plan->host_call.reset();
    plan->host_bytes = 0;
    return SDDMM_OK;
}
