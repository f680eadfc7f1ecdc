// Error reporting and version of the C ABI.
#include "common.hpp"

#include <atomic>
#include <chrono>
#include <mutex>

namespace mstf {
static std::atomic<int> g_last_hip_error{0};
void set_last_hip_error(int e) { g_last_hip_error.store(e); }

// Polls a one-pass producer's workgroup spends on a wait before it gives up (0 in the atomic = the default).
static std::atomic<uint32_t> g_spin_limit{0u};
static std::atomic<bool> g_spin_limit_set{false};
uint32_t onepass_spin_limit() { return g_spin_limit_set.load() ? g_spin_limit.load() : (1u << 20); }
}  // namespace mstf

extern "C" void mstf_test_set_spin_limit(int64_t polls)
{
    if (polls < 0) {
        mstf::g_spin_limit_set.store(false);
        return;
    }
    mstf::g_spin_limit.store(polls > 0xFFFFFFFFll ? 0xFFFFFFFFu : (uint32_t)polls);
    mstf::g_spin_limit_set.store(true);
}

extern "C" const char* mstf_strerror(int code)
{
    switch (code) {
        case MSTF_OK: return "ok";
        case MSTF_EINVAL: return "invalid argument (null pointer, non-positive size or inconsistent shape)";
        case MSTF_EALIGN: return "pointer not aligned as required";
        case MSTF_EUNSUPPORTED: return "shape not supported by the gfx950 kernels";
        case MSTF_EWORKSPACE: return "workspace missing or too small";
        case MSTF_ELAUNCH: return "HIP kernel launch failed (see mstf_last_hip_error)";
        case MSTF_ETOOLARGE:
            return "the problem needs more scratch memory than the library's fixed buffer holds (use the entry point "
                   "that takes a workspace)";
        default: return "unknown error code";
    }
}

extern "C" int mstf_last_hip_error(void) { return mstf::g_last_hip_error.load(); }

extern "C" int mstf_version(void) { return 100; }

// ------------------------------------------------------------------ measurement aid
// Streams `bytes` of device memory with 16-byte loads per lane and nothing else (the xor of everything read goes to
// sink[workgroup]): the plain-read time of a buffer, against which the kernels' times are read.
namespace mstf {
__global__ __launch_bounds__(256) void read_probe_kernel(const uint4* __restrict__ src, size_t n16, uint32_t* __restrict__ sink)
{
    uint4 acc = {0u, 0u, 0u, 0u};
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride) {
        const uint4 v = src[i];
        acc.x ^= v.x;
        acc.y ^= v.y;
        acc.z ^= v.z;
        acc.w ^= v.w;
    }
    const uint32_t r = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (r == 0x9e3779b9u) sink[blockIdx.x] = r;  // practically never: keeps the loads alive without a store per lane
}
}  // namespace mstf

extern "C" int mstf_probe_read(void* stream, const void* src, size_t bytes, uint32_t* sink, int workgroups)
{
    if (!src || !sink || bytes < 16 || workgroups <= 0) return MSTF_EINVAL;
    if (!mstf::aligned_to(src, 16) || !mstf::aligned_to(sink, 4)) return MSTF_EALIGN;
    hipLaunchKernelGGL(mstf::read_probe_kernel, dim3((unsigned)workgroups), dim3(256), 0, mstf::as_stream(stream),
                       reinterpret_cast<const uint4*>(src), bytes / 16, sink);
    return mstf::check_launch();
}

// ------------------------------------------------------------------ a word on the host
// What a caller who sizes its next step by a result pays between the end of the kernels and its own next line: a copy to the
// host and a stream synchronisation take 12.7 us on an idle stream, a store to pinned memory that the thread watches 7.2 us.
namespace mstf {
__global__ void publish_word_kernel(const int64_t* __restrict__ src, int64_t* landing)
{
    __hip_atomic_store(landing, *src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace mstf

int mstf::stream_recorded(hipStream_t st, bool* recorded)
{
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(st, &capturing);
    if (e != hipSuccess) {
        set_last_hip_error((int)e);
        return MSTF_ELAUNCH;
    }
    *recorded = capturing != hipStreamCaptureStatusNone;
    return MSTF_OK;
}

int mstf::landing_ready(hipStream_t st, int64_t* landing, const int64_t* value)
{
    if (!landing || !value) return MSTF_EINVAL;
    if (!aligned_to(landing, 8)) return MSTF_EALIGN;
    bool recorded = false;
    const int rc = stream_recorded(st, &recorded);
    if (rc != MSTF_OK) return rc;
    if (recorded) {
        set_last_hip_error((int)hipErrorStreamCaptureUnsupported);
        return MSTF_ELAUNCH;
    }
    __atomic_store_n(landing, kLandingEmpty, __ATOMIC_RELEASE);
    return MSTF_OK;
}

int mstf::landing_wait(hipStream_t st, const int64_t* landing, int64_t* value)
{
    // Long waits (a full stream, an error that keeps the word from coming) are left to the runtime.
    constexpr auto kWatch = std::chrono::microseconds(500);
    const auto until = std::chrono::steady_clock::now() + kWatch;
    int64_t v = kLandingEmpty;
    do {
        for (int i = 0; i < 64 && v == kLandingEmpty; i++) v = __atomic_load_n(landing, __ATOMIC_ACQUIRE);
    } while (v == kLandingEmpty && std::chrono::steady_clock::now() < until);
    if (v == kLandingEmpty) {
        bool recorded = false;
        const int rc = stream_recorded(st, &recorded);
        if (rc != MSTF_OK) return rc;
        const hipError_t e = recorded ? hipErrorStreamCaptureUnsupported : hipStreamSynchronize(st);
        if (e != hipSuccess) {
            set_last_hip_error((int)e);
            return MSTF_ELAUNCH;
        }
        v = __atomic_load_n(landing, __ATOMIC_ACQUIRE);
    }
    *value = v;
    return MSTF_OK;
}

int mstf::total_wait(hipStream_t st, const int64_t* landing, int64_t* value)
{
    const int rc = landing_wait(st, landing, value);
    if (rc != MSTF_OK || *value != kLandingEmpty) return rc;
    set_last_hip_error((int)hipErrorNotReady);  // the stream is done and nothing has come
    return MSTF_ELAUNCH;
}

extern "C" int mstf_read_word(void* stream, const int64_t* src, int64_t* landing, int64_t* value)
{
    if (!src || !landing || !value) return MSTF_EINVAL;
    if (!mstf::aligned_to(src, 8) || !mstf::aligned_to(landing, 8)) return MSTF_EALIGN;
    hipStream_t st = mstf::as_stream(stream);
    int rc = mstf::landing_ready(st, landing, value);
    if (rc != MSTF_OK) return rc;
    hipLaunchKernelGGL(mstf::publish_word_kernel, dim3(1), dim3(1), 0, st, src, landing);
    rc = mstf::check_launch();
    return rc != MSTF_OK ? rc : mstf::landing_wait(st, landing, value);
}

extern "C" int mstf_landing_wait(void* stream, const int64_t* landing, int64_t* value)
{
    if (!landing || !value) return MSTF_EINVAL;
    if (!mstf::aligned_to(landing, 8)) return MSTF_EALIGN;
    return mstf::total_wait(mstf::as_stream(stream), landing, value);
}

// ------------------------------------------------------------------ landings of calls that are not waited for
// Pairs of words in one block of pinned memory, made with the first of them and kept: 1024 pairs, so that a program that holds
// on to more results than that finds none free and reads its totals by mstf_read_word.  A pair that is given back while its
// kernel has yet to store to it stays away from the others until it has.  The first call may be one that is being recorded: the
// allocation is no part of what is recorded, and a failure leaves no error for the launch behind it to find.
namespace mstf {
static std::mutex g_landing_lock;
static int64_t* g_landing_block = nullptr;
static bool g_landing_failed = false;
constexpr int kLandingPairs = 1024;
static uint16_t g_landing_free[kLandingPairs];  // a ring: the one that was given back first is the first to be taken
static bool g_landing_taken[kLandingPairs];
static int g_landing_head = 0, g_landing_count = 0;
}  // namespace mstf

extern "C" int64_t* mstf_landing_take(void)
{
    using namespace mstf;
    std::lock_guard<std::mutex> hold(g_landing_lock);
    if (!g_landing_block) {
        if (g_landing_failed) return nullptr;
        void* p = nullptr;
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // (of this thread, for this call alone)
        const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
        const hipError_t e = hipHostMalloc(&p, kLandingPairs * 2 * sizeof(int64_t), hipHostMallocPortable | hipHostMallocMapped);
        if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            // (refused because of a capture somewhere: asked again by the next call)
            g_landing_failed = e != hipErrorStreamCaptureUnsupported && e != hipErrorStreamCaptureImplicit;
            return nullptr;
        }
        g_landing_block = static_cast<int64_t*>(p);
        for (int i = 0; i < kLandingPairs; i++) {
            g_landing_block[2 * i] = g_landing_block[2 * i + 1] = MSTF_NOT_LANDED;
            g_landing_free[i] = (uint16_t)i;
        }
        g_landing_count = kLandingPairs;
    }
    if (g_landing_count == 0) return nullptr;
    const uint16_t at = g_landing_free[g_landing_head];
    int64_t* pair = g_landing_block + 2 * at;
    for (int i = 0; i < 2; i++)
        if (__atomic_load_n(pair + i, __ATOMIC_ACQUIRE) == kLandingEmpty) return nullptr;  // (and those behind it are younger)
    g_landing_head = (g_landing_head + 1) % kLandingPairs;
    g_landing_count--;
    g_landing_taken[at] = true;
    return pair;
}

extern "C" void mstf_landing_give(int64_t* pair)
{
    using namespace mstf;
    std::lock_guard<std::mutex> hold(g_landing_lock);
    if (!pair || !g_landing_block || pair < g_landing_block || pair >= g_landing_block + 2 * kLandingPairs) return;
    const uint16_t at = (uint16_t)((pair - g_landing_block) / 2);
    if (pair != g_landing_block + 2 * at || !g_landing_taken[at]) return;  // no pair, or not out
    g_landing_taken[at] = false;
    g_landing_free[(g_landing_head + g_landing_count) % kLandingPairs] = at;
    g_landing_count++;
}
