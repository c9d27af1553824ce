// A stand-in for the HIP runtime on the host, enough of it to run the library's copies (transfer.hip, runtime.hip) without a GPU:
// streams are threads that work their queues off in order, device memory is host memory, the two copy kernels are memcpy. A copy
// takes `g_copy_us` before it touches its bytes, so that whatever reuses them too early is seen.
#include "host_device.h"

#include <condition_variable>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>

#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

std::atomic<int> g_copy_us{0}, g_mallocs{0}, g_malloc_us{0};
std::atomic<bool> g_no_threads{false};

// libstdc++'s threads come through here
extern "C" int pthread_create(pthread_t* thread, const pthread_attr_t* attr, void* (*start)(void*), void* arg) {
    static const auto real = reinterpret_cast<int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*)>(dlsym(RTLD_NEXT, "pthread_create"));
    return g_no_threads ? EAGAIN : real(thread, attr, start, arg);
}

struct ihipStream_t {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> queue;
    bool busy = false, closing = false;
    std::thread worker;
    ihipStream_t() : worker([this] { work(); }) {}
    ~ihipStream_t() {
        {
            std::lock_guard<std::mutex> g(mu);
            closing = true;
        }
        cv.notify_all();
        worker.join();
    }
    void work() {
        std::unique_lock<std::mutex> g(mu);
        for (;;) {
            cv.wait(g, [this] { return closing || !queue.empty(); });
            if (queue.empty()) return;
            auto f = std::move(queue.front());
            queue.pop_front();
            busy = true;
            g.unlock();
            f();
            g.lock();
            busy = false;
            cv.notify_all();
        }
    }
    void push(std::function<void()> f) {
        {
            std::lock_guard<std::mutex> g(mu);
            queue.push_back(std::move(f));
        }
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> g(mu);
        cv.wait(g, [this] { return queue.empty() && !busy; });
    }
};

struct ihipEvent_t {
    std::mutex mu;
    std::condition_variable cv;
    long recorded = 0, reached = 0;
    void wait_for(long n) {
        std::unique_lock<std::mutex> g(mu);
        cv.wait(g, [&] { return reached >= n; });
    }
};

namespace {
std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> names;
    return names;
}
struct call_config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local call_config t_call;
void copy(void* dst, const void* src, size_t bytes) {
    if (g_copy_us) usleep(g_copy_us);
    memcpy(dst, src, bytes);
}
}  // namespace

extern "C" {
char __hip_fatbin = 0;
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels()[host] = name; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    t_call = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = t_call.grid;
    *block = t_call.block;
    *shared = t_call.shared;
    *stream = t_call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t stream) {
    const std::string& name = kernels().at(f);
    const char* src = *static_cast<const char**>(args[0]);
    char* dst = *static_cast<char**>(args[1]);
    const unsigned bytes = *static_cast<unsigned*>(args[2]);
    if (name.find("download_kernel") == std::string::npos) {
        stream->push([=] { copy(dst, src, bytes); });
    } else {
        unsigned* flag = *static_cast<unsigned**>(args[4]);
        const unsigned value = *static_cast<unsigned*>(args[5]);
        stream->push([=] {
            copy(dst, src, bytes);
            __atomic_store_n(flag, value, __ATOMIC_RELEASE);
        });
    }
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) { return *s = new ihipStream_t, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return delete s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return s->wait(), hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::unique_lock<std::mutex> g(e->mu);
    const long n = e->recorded;
    g.unlock();
    s->push([=] { e->wait_for(n); });
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return *e = new ihipEvent_t, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::unique_lock<std::mutex> g(e->mu);
    const long n = ++e->recorded;
    g.unlock();
    s->push([=] {
        std::lock_guard<std::mutex> h(e->mu);
        e->reached = n;
        e->cv.notify_all();
    });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::unique_lock<std::mutex> g(e->mu);
    const long n = e->recorded;
    g.unlock();
    return e->wait_for(n), hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipMalloc(void** p, size_t bytes) {
    ++g_mallocs;
    if (g_malloc_us) usleep(g_malloc_us);
    *p = aligned_alloc(256, (bytes + 255) / 256 * 256);
    return hipSuccess;
}
hipError_t hipFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return *p = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096), hipSuccess; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s) { return s->push([=] { copy(dst, src, bytes); }), hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t bytes) { return memset(p, v, bytes), hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t bytes, hipStream_t s) { return s->push([=] { memset(p, v, bytes); }), hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { return *s = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

int exhip_static_scratch_setup(int) { return 0; }
