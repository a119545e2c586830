// common.hip -- error state, lazy device init, pointer checks, scratch.
#include "common.hpp"

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

namespace gfh {

namespace {
thread_local std::string g_last_error = "No error";
std::atomic<int> g_pointer_checks{1};
std::once_flag g_init_once;
int g_init_status = GFH_UNKNOWN;
std::string g_init_message;
}  // namespace

int set_error(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

void clear_error() { g_last_error = "No error"; }

const char *last_error() { return g_last_error.c_str(); }

int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(GFH_COMPUTATION_FAILED, "%s: launch failed: %s", what, hipGetErrorString(e));
    return GFH_SUCCESS;
}

int ensure_init() {
    std::call_once(g_init_once, [] {
        int n = 0;
        hipError_t e = hipGetDeviceCount(&n);
        if (e != hipSuccess || n == 0) {
            g_init_status = GFH_COMPUTATION_FAILED;
            g_init_message = std::string("no HIP device available: ") +
                             (e != hipSuccess ? hipGetErrorString(e) : "device count is 0");
            return;
        }
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) {
            g_init_status = GFH_COMPUTATION_FAILED;
            g_init_message = "hipGetDevice failed";
            return;
        }
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) {
            g_init_status = GFH_COMPUTATION_FAILED;
            g_init_message = "hipGetDeviceProperties failed";
            return;
        }
        if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
            g_init_status = GFH_COMPUTATION_FAILED;
            g_init_message = std::string("kernels are built for gfx950, device is ") + prop.gcnArchName;
            return;
        }
        g_init_status = GFH_SUCCESS;
    });
    if (g_init_status != GFH_SUCCESS) return set_error(g_init_status, "%s", g_init_message.c_str());
    return GFH_SUCCESS;
}

int check_device_ptr(const void *p, const char *name) {
    if (!g_pointer_checks.load(std::memory_order_relaxed)) return GFH_SUCCESS;
    hipPointerAttribute_t attr;
    hipError_t e = hipPointerGetAttributes(&attr, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // do not leave the lookup failure for the next launch check
        return set_error(GFH_INVALID_DATA, "%s is not a device pointer (%s)", name, hipGetErrorString(e));
    }
    if (attr.type != hipMemoryTypeDevice && attr.type != hipMemoryTypeManaged)
        return set_error(GFH_INVALID_DATA, "%s is not device memory (memory type %d)", name, (int)attr.type);
    return GFH_SUCCESS;
}

int require_ptr(const void *p, const char *name) {
    if (!p) return set_error(GFH_NULL_POINTER, "%s is NULL", name);
    return check_device_ptr(p, name);
}

int require_range(const void *p, size_t bytes, const char *name) {
    if (!p) {
        if (bytes == 0) return GFH_SUCCESS;
        return set_error(GFH_NULL_POINTER, "%s is NULL", name);
    }
    if (!g_pointer_checks.load(std::memory_order_relaxed)) return GFH_SUCCESS;
    GFH_TRY(check_device_ptr(p, name));
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    hipError_t e = hipMemGetAddressRange(&base, &size, const_cast<void *>(p));
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return set_error(GFH_INVALID_DATA, "%s: no device allocation contains this address (%s)", name,
                         hipGetErrorString(e));
    }
    const uintptr_t lo = reinterpret_cast<uintptr_t>(base);
    const uintptr_t hi = lo + size;
    const uintptr_t at = reinterpret_cast<uintptr_t>(p);
    if (at < lo || bytes > hi - at)
        return set_error(GFH_INVALID_SHAPE, "%s: %zu bytes needed but only %zu remain in its allocation", name,
                         bytes, (size_t)(hi - at));
    return GFH_SUCCESS;
}

int optional_range(const void *p, size_t bytes, const char *name) {
    if (!p) return GFH_SUCCESS;
    return require_range(p, bytes, name);
}

namespace {

// Zeroes a new counter buffer on its stream.  A fill kernel rather than
// hipMemsetAsync: where a stream is captured into a graph, memset nodes have
// given wrong results on replays after the first.
__global__ void zero_counters_kernel(int *p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// The library's per-stream buffers (and stream-ordered scratch) are
// allocated on first use.  On a stream that is being captured into a graph
// that allocation would become part of the graph, so it is refused: the
// caller runs the call once on the stream before capturing it (or passes a
// workspace), and the captured calls then allocate nothing.
int refuse_during_capture(hipStream_t s, const char *what) {
    if (s == nullptr) return GFH_SUCCESS;  // the legacy default stream is never captured
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return GFH_SUCCESS;
    }
    if (st != hipStreamCaptureStatusNone)
        return set_error(GFH_ALLOCATION_FAILED,
                         "%s: the stream is being captured into a graph; run the call once on this stream before "
                         "capturing it (per-stream buffers are allocated on first use) or pass a workspace",
                         what);
    return GFH_SUCCESS;
}

}  // namespace

namespace {

// Scratch blocks kept between calls, one per (device, stream): the calls of
// a stream run in order, so the next one may write where the last one's
// kernels still read.  A block serves one call at a time; a second thread
// issuing on the same stream meanwhile allocates its own.
struct ScratchBlock {
    void *p = nullptr;
    size_t bytes = 0;
    bool busy = false;
    uint64_t last = 0;          // g_block_calls when it was last taken
    hipEvent_t done = nullptr;  // after its last use, where `recorded`
    bool recorded = false;
};
// Needs above kBlockMax, and blocks past kBlockTotal over all streams, are
// allocated and freed per call: there the kernels outlast the ~17 us of host
// time that hipMallocAsync and hipFreeAsync take (INT8 dynamic linear, 100 x
// 4096 x 11008, 21 us of kernels: 25 to 30 us per call of the C entry with
// them, 21 without).
constexpr size_t kBlockMax = (size_t)64 << 20, kBlockTotal = (size_t)256 << 20;
// Nothing tells when a stream is destroyed, so a block goes to another stream
// once kBlockIdle calls have passed it by and the total leaves no other room.
// The new owner waits for an event that the old stream recorded after its last
// use; blocks record one from half the total on, so that programs with a few
// streams do not pay for it.
constexpr uint64_t kBlockIdle = 256;
std::mutex g_block_mu;
std::map<std::pair<int, hipStream_t>, ScratchBlock> g_blocks;
size_t g_block_bytes = 0;
uint64_t g_block_calls = 0;

// Drops idle blocks of the device, the longest unused first, until `want` more
// bytes fit the total: frees them in the order of s.  False when they do not.
bool make_room(int dev, size_t want, hipStream_t s) {
    while (g_block_bytes + want > kBlockTotal) {
        auto oldest = g_blocks.end();
        for (auto it = g_blocks.begin(); it != g_blocks.end(); ++it) {
            const ScratchBlock &b = it->second;
            if (it->first.first != dev || it->first.second == s || b.busy || !b.recorded ||
                g_block_calls - b.last < kBlockIdle)
                continue;
            if (oldest == g_blocks.end() || b.last < oldest->second.last) oldest = it;
        }
        if (oldest == g_blocks.end()) return false;
        ScratchBlock &b = oldest->second;
        if (hipStreamWaitEvent(s, b.done, 0) != hipSuccess || hipFreeAsync(b.p, s) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        (void)hipEventDestroy(b.done);
        g_block_bytes -= b.bytes;
        g_blocks.erase(oldest);
    }
    return true;
}

// The stream's block, taken for the caller, or null where there is none to
// have (the caller then allocates).
void *take_block(int dev, size_t need, hipStream_t s) {
    // (hipStreamPerThread names a different stream in every thread)
    if (need > kBlockMax || s == hipStreamPerThread) return nullptr;
    std::lock_guard<std::mutex> lock(g_block_mu);
    ++g_block_calls;
    ScratchBlock &b = g_blocks[std::make_pair(dev, s)];
    if (b.busy) return nullptr;
    if (b.bytes < need) {
        size_t want = (size_t)1 << 20;
        while (want < need) want *= 2;
        if (!make_room(dev, want - b.bytes, s)) return nullptr;
        void *p = nullptr;
        if (hipMallocAsync(&p, want, s) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (b.p) (void)hipFreeAsync(b.p, s);
        g_block_bytes += want - b.bytes;
        b.p = p;
        b.bytes = want;
    }
    b.busy = true;
    b.recorded = false;
    b.last = g_block_calls;
    return b.p;
}

void return_block(int dev, hipStream_t s) {
    std::lock_guard<std::mutex> lock(g_block_mu);
    ScratchBlock &b = g_blocks[std::make_pair(dev, s)];
    b.busy = false;
    if (g_block_bytes <= kBlockTotal / 2) return;
    if (!b.done && hipEventCreateWithFlags(&b.done, hipEventDisableTiming) != hipSuccess) b.done = nullptr;
    b.recorded = b.done && hipEventRecord(b.done, s) == hipSuccess;
    if (!b.recorded) (void)hipGetLastError();
}

// Frees the blocks that no call holds.
void release_blocks() {
    std::lock_guard<std::mutex> lock(g_block_mu);
    if (g_blocks.empty()) return;
    (void)hipDeviceSynchronize();
    for (auto it = g_blocks.begin(); it != g_blocks.end();) {
        if (it->second.busy) {
            ++it;
            continue;
        }
        if (it->second.p) (void)hipFree(it->second.p);
        if (it->second.done) (void)hipEventDestroy(it->second.done);
        g_block_bytes -= it->second.bytes;
        it = g_blocks.erase(it);
    }
}

}  // namespace

Scratch::~Scratch() {
    if (dev_ >= 0)
        return_block(dev_, s_);
    else if (owned_ && p_)
        (void)hipFreeAsync(p_, s_);
}

int Scratch::acquire(void *user, size_t user_bytes, size_t need, hipStream_t s) {
    if (need == 0) need = 16;
    if (user) {
        if (user_bytes < need)
            return set_error(GFH_INVALID_SHAPE, "workspace of %zu bytes is smaller than the %zu required",
                             user_bytes, need);
        GFH_TRY(check_device_ptr(user, "workspace"));
        p_ = user;
        owned_ = false;
        return GFH_SUCCESS;
    }
    GFH_TRY(refuse_during_capture(s, "workspace"));
    s_ = s;
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess && (p_ = take_block(dev, need, s)) != nullptr) {
        dev_ = dev;
        return GFH_SUCCESS;
    }
    hipError_t e = hipMallocAsync(&p_, need, s);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        p_ = nullptr;
        return set_error(GFH_ALLOCATION_FAILED, "hipMallocAsync(%zu) failed: %s", need, hipGetErrorString(e));
    }
    owned_ = true;
    return GFH_SUCCESS;
}

namespace {
struct StreamState {
    int *counters = nullptr;
    size_t ncounters = 0;
    void *ws = nullptr;
    size_t ws_bytes = 0;
};
std::mutex g_state_mu;
std::map<std::pair<int, hipStream_t>, StreamState> g_states;
std::vector<void *> g_retired;  // outgrown buffers (maybe still in use by queued work), freed at shutdown

int current_state(hipStream_t s, StreamState **out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return set_error(GFH_COMPUTATION_FAILED, "hipGetDevice failed");
    }
    *out = &g_states[std::make_pair(dev, s)];
    return GFH_SUCCESS;
}
}  // namespace

int stream_counters(hipStream_t s, size_t count, int **out) {
    std::lock_guard<std::mutex> lock(g_state_mu);
    StreamState *st = nullptr;
    GFH_TRY(current_state(s, &st));
    if (st->ncounters < count) {
        GFH_TRY(refuse_during_capture(s, "split-K counters"));
        size_t want = 4096;
        while (want < count) want *= 2;
        int *p = nullptr;
        hipError_t e = hipMallocAsync(reinterpret_cast<void **>(&p), want * sizeof(int), s);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(zero_counters_kernel, dim3((unsigned)((want + 255) / 256)), dim3(256), 0, s, p, want);
            e = hipGetLastError();
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return set_error(GFH_ALLOCATION_FAILED, "counter buffer allocation failed: %s", hipGetErrorString(e));
        }
        if (st->counters) g_retired.push_back(st->counters);
        st->counters = p;
        st->ncounters = want;
    }
    *out = st->counters;
    return GFH_SUCCESS;
}

int device_cu_count() {
    constexpr int kMaxDevices = 64;
    static std::atomic<int> cache[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
    int n = cache[dev].load(std::memory_order_relaxed);
    if (n > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
    return n;
}

int stream_workspace(hipStream_t s, size_t bytes, void **out) {
    std::lock_guard<std::mutex> lock(g_state_mu);
    StreamState *st = nullptr;
    GFH_TRY(current_state(s, &st));
    if (st->ws_bytes < bytes) {
        GFH_TRY(refuse_during_capture(s, "split-K workspace"));
        size_t want = (size_t)1 << 20;
        while (want < bytes) want *= 2;
        void *p = nullptr;
        hipError_t e = hipMallocAsync(&p, want, s);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return set_error(GFH_ALLOCATION_FAILED, "workspace allocation (%zu bytes) failed: %s", want,
                             hipGetErrorString(e));
        }
        if (st->ws) g_retired.push_back(st->ws);
        st->ws = p;
        st->ws_bytes = want;
    }
    *out = st->ws;
    return GFH_SUCCESS;
}

void release_stream_state() {
    release_blocks();
    std::lock_guard<std::mutex> lock(g_state_mu);
    if (g_states.empty() && g_retired.empty()) return;
    (void)hipDeviceSynchronize();
    for (auto &kv : g_states) {
        if (kv.second.counters) (void)hipFree(kv.second.counters);
        if (kv.second.ws) (void)hipFree(kv.second.ws);
    }
    for (void *p : g_retired) (void)hipFree(p);
    g_states.clear();
    g_retired.clear();
}

int set_pointer_checks(int enabled) {
    g_pointer_checks.store(enabled ? 1 : 0);
    return GFH_SUCCESS;
}

}  // namespace gfh

// Bytes kept for the current device's stream s.  Not part of the API: for the
// tests.
extern "C" __attribute__((visibility("default"))) size_t gfh_internal_scratch_kept(hipStream_t s) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(gfh::g_block_mu);
    const auto it = gfh::g_blocks.find(std::make_pair(dev, s));
    return it == gfh::g_blocks.end() ? 0 : it->second.bytes;
}
