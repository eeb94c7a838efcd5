// Uploads of host arrays: through pinned memory, by several threads, overlapped with the transfer.
//
// A copy from pageable memory runs at 38 GB/s on a machine whose link moves 57 (38.5 MB, ResNet-18 at batch 64: 1008 us
// against 678 from pinned memory), and the scan for max |x| that guards the residual formats was another pass over the
// array (632 us there, 244 us for 2.4 MB).  Here one pass copies a piece into pinned memory and takes its maximum, the
// pieces are shared with a few worker threads, and chunks go to the device as they fill up; the transfer is then all that
// is left (set_input of 38.5 MB 1961 -> 800 us, of 2.4 MB 346 -> 92, of 0.6 MB 96 -> 45).
// An uploader has to be made first, and the pages of its pinned memory are slow when they are first written (38.5 MB: 0.9 ms
// and 3.5 ms), so the layers make one for their second batch, not for the first.  (16 MiB of pinned memory, used as a ring or
// in two halves, cost 2 ms less there, and 90 to 260 us on every batch of 38.5 MB after it.)
#include <hip/hip_runtime_api.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include "../../include/tcbnn_hip.h"

namespace tcbnn {
int fail(int code, const char* fmt, ...);
int check_hip(hipError_t e, const char* what);
}  // namespace tcbnn

namespace {

constexpr size_t kPiece = 128 << 10;       // bytes a thread takes at a time
constexpr size_t kPinnedMost = 64 << 20;   // pinned memory per uploader; longer arrays go through it in turns
constexpr size_t kOverlapFrom = 4 << 20;   // from here on chunks are transferred while later ones are copied
constexpr size_t kFirstChunk = 384 << 10;  // each further chunk is three times as long: a transfer costs 9 us whatever its length
// From here on (half a last-level cache) the copy writes past the caches: it then leaves the memory to the transfer beside
// it (38.5 MB staged in 957 us with ordinary stores, 757 us with these; 8.4 MB in 197 and 212 us).
constexpr size_t kStreamFrom = 16 << 20;
constexpr int kMostWorkers = 7;

// The largest bit pattern of |x|: patterns of finite magnitudes order as the magnitudes, infinities and NaNs lie above.
uint32_t copy_max_plain(uint32_t* dst, const uint32_t* src, size_t n) {
    uint32_t m = 0;
    for (size_t i = 0; i < n; ++i) {
        const uint32_t v = src[i], a = v & 0x7fffffffu;
        if (dst != nullptr) dst[i] = v;
        m = a > m ? a : m;
    }
    return m;
}
#if defined(__x86_64__)
template <bool STREAM>
__attribute__((target("avx2"))) uint32_t copy_max_avx2(uint32_t* dst, const uint32_t* src, size_t n) {
    const __m256i mask = _mm256_set1_epi32(0x7fffffff);
    __m256i m[4] = {_mm256_setzero_si256(), _mm256_setzero_si256(), _mm256_setzero_si256(), _mm256_setzero_si256()};
    size_t i = 0;
    for (; i + 32 <= n; i += 32)
        for (int k = 0; k < 4; ++k) {
            const __m256i v = _mm256_loadu_si256(reinterpret_cast<const __m256i*>(src + i + 8 * k));
            if (STREAM) _mm256_stream_si256(reinterpret_cast<__m256i*>(dst + i + 8 * k), v);  // (pinned memory: aligned)
            else if (dst != nullptr) _mm256_storeu_si256(reinterpret_cast<__m256i*>(dst + i + 8 * k), v);
            m[k] = _mm256_max_epu32(m[k], _mm256_and_si256(v, mask));
        }
    if (STREAM) _mm_sfence();
    uint32_t lanes[8];
    _mm256_storeu_si256(reinterpret_cast<__m256i*>(lanes), _mm256_max_epu32(_mm256_max_epu32(m[0], m[1]), _mm256_max_epu32(m[2], m[3])));
    const uint32_t rest = copy_max_plain(dst != nullptr ? dst + i : nullptr, src + i, n - i);
    return std::max(rest, *std::max_element(lanes, lanes + 8));
}
#endif
uint32_t copy_max(uint32_t* dst, const uint32_t* src, size_t n, bool stream) {
#if defined(__x86_64__)
    static const bool avx2 = __builtin_cpu_supports("avx2");
    if (avx2) return stream && dst != nullptr ? copy_max_avx2<true>(dst, src, n) : copy_max_avx2<false>(dst, src, n);
#endif
    return copy_max_plain(dst, src, n);
}
float magnitude(uint32_t pattern) {
    float f;
    memcpy(&f, &pattern, 4);
    return f <= 3.0e38f ? f : INFINITY;  // (NaN or infinity anywhere: +infinity)
}

// One pass over an array, in pieces that any thread may take; chunks are runs of pieces.
struct Job {
    char* dst = nullptr;
    const char* src = nullptr;
    size_t bytes = 0;
    std::atomic<size_t> next{0};
    std::atomic<uint32_t> most{0};
    std::vector<size_t> chunk_end;                 // in pieces
    std::unique_ptr<std::atomic<size_t>[]> left;   // pieces of each chunk still to copy
    size_t pieces() const { return (bytes + kPiece - 1) / kPiece; }
    // takes one piece; false when none is left
    bool work() {
        const size_t p = next.fetch_add(1, std::memory_order_relaxed);
        if (p >= pieces()) return false;
        const size_t at = p * kPiece, n = std::min(kPiece, bytes - at);
        const uint32_t m = copy_max(reinterpret_cast<uint32_t*>(dst + at), reinterpret_cast<const uint32_t*>(src + at), n / 4,
                                    bytes >= kStreamFrom);
        if (n % 4 != 0) memcpy(dst + at + n / 4 * 4, src + at + n / 4 * 4, n % 4);
        uint32_t seen = most.load(std::memory_order_relaxed);
        while (m > seen && !most.compare_exchange_weak(seen, m, std::memory_order_relaxed)) {
        }
        size_t c = 0;
        while (p >= chunk_end[c]) ++c;
        left[c].fetch_sub(1, std::memory_order_release);
        return true;
    }
};

// Up to n threads that run `work`: as many as can be had, none at worst (a limit on threads or memory is no reason to give
// up what the caller can do alone, and a half-filled vector of running threads must not be destroyed).
template <class F>
std::vector<std::thread> start_threads(int n, F work) {
    std::vector<std::thread> t;
    try {
        t.reserve((size_t)std::max(0, n));
        while ((int)t.size() < n) t.emplace_back(work);
    } catch (const std::exception&) {
    }
    return t;
}

// Worker threads, shared by all uploaders of the process and gone with the last of them.  One job at a time; a caller that
// finds them busy does its job alone.
class Workers {
  public:
    static std::shared_ptr<Workers> get() {
        static std::mutex guard;
        static std::weak_ptr<Workers> one;
        std::lock_guard<std::mutex> l(guard);
        std::shared_ptr<Workers> w = one.lock();
        if (!w) one = w = std::make_shared<Workers>();
        return w;
    }
    Workers() : threads_(start_threads(std::min(kMostWorkers, (int)std::thread::hardware_concurrency() - 1), [this] { loop(); })) {}
    ~Workers() {
        {
            std::lock_guard<std::mutex> l(m_);
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread& t : threads_) t.join();
    }
    bool start(Job* job) {
        if (!owner_.try_lock()) return false;
        {
            std::lock_guard<std::mutex> l(m_);
            job_ = job;
            ++round_;
        }
        wake_.notify_all();
        return true;
    }
    void finish() {  // (every piece has been taken; waits for the threads that still hold one)
        {
            std::unique_lock<std::mutex> l(m_);
            job_ = nullptr;
            idle_.wait(l, [this] { return inside_ == 0; });
        }
        owner_.unlock();
    }

  private:
    void loop() {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> l(m_);
        for (;;) {
            wake_.wait(l, [&] { return stop_ || (job_ != nullptr && round_ != seen); });
            if (stop_) return;
            seen = round_;
            Job* job = job_;
            ++inside_;
            l.unlock();
            while (job->work()) {
            }
            l.lock();
            if (--inside_ == 0) idle_.notify_all();
        }
    }
    std::mutex owner_, m_;
    std::condition_variable wake_, idle_;
    Job* job_ = nullptr;
    uint64_t round_ = 0;
    int inside_ = 0;
    bool stop_ = false;
    std::vector<std::thread> threads_;  // (last: started when all that they use is there)
};

}  // namespace

using tcbnn::check_hip;
using tcbnn::fail;

struct tcbnn_uploader {
    std::mutex m;
    size_t bytes = 0, pinned_bytes = 0;
    void* pinned = nullptr;
    void* device = nullptr;  // where a staged array waits for its commit
    bool on_device = false;  // the staged array is there (else in pinned memory)
    size_t staged = 0;
    std::shared_ptr<Workers> workers;
    ~tcbnn_uploader() {
        if (device != nullptr) (void)hipFree(device);
        if (pinned != nullptr) (void)hipHostFree(pinned);
    }
};

namespace {

// Copies `bytes` of `src` into the pinned memory and, where `to` is given, on to the device, chunk by chunk on the null
// stream (the order a plain copy has).  The pinned memory is free again, and the maximum final, when it returns.
int pass(tcbnn_uploader* u, void* to, const void* src, size_t bytes, uint32_t* most) {
    for (size_t at = 0; at < bytes; at += u->pinned_bytes) {
        Job job;
        job.bytes = std::min(u->pinned_bytes, bytes - at);
        job.src = static_cast<const char*>(src) + at;
        job.dst = static_cast<char*>(u->pinned);
        size_t chunk = to != nullptr && job.bytes >= kOverlapFrom ? kFirstChunk : job.bytes;
        for (size_t end = 0; end < job.bytes; chunk *= 3) {
            end = std::min(end + chunk, job.bytes);
            job.chunk_end.push_back((end + kPiece - 1) / kPiece);
        }
        const size_t chunks = job.chunk_end.size();
        job.left.reset(new std::atomic<size_t>[chunks]);
        for (size_t c = 0; c < chunks; ++c) job.left[c] = job.chunk_end[c] - (c > 0 ? job.chunk_end[c - 1] : 0);

        const bool shared = job.bytes > 4 * kPiece && u->workers && u->workers->start(&job);
        int rc = TCBNN_OK;
        for (size_t c = 0; c < chunks; ++c) {
            while (job.left[c].load(std::memory_order_acquire) != 0)
                if (!job.work()) std::this_thread::yield();
            if (to != nullptr && rc == TCBNN_OK) {
                const size_t b = (c > 0 ? job.chunk_end[c - 1] : 0) * kPiece, e = std::min(job.chunk_end[c] * kPiece, job.bytes);
                rc = check_hip(hipMemcpyAsync(static_cast<char*>(to) + at + b, static_cast<char*>(u->pinned) + b, e - b,
                                              hipMemcpyHostToDevice, nullptr),
                               "hipMemcpyAsync H2D");
            }
        }
        if (shared) u->workers->finish();
        if (to != nullptr)
            if (int e = check_hip(hipStreamSynchronize(nullptr), "hipStreamSynchronize")) rc = rc != TCBNN_OK ? rc : e;
        if (rc != TCBNN_OK) return rc;
        if (most != nullptr) *most = std::max(*most, job.most.load());
    }
    return TCBNN_OK;
}

}  // namespace

extern "C" {

// (no exception leaves an entry point: allocations of the host side that fail are an error code)
static int out_of_memory(const char* what) { return fail(TCBNN_EINVAL, "%s: out of host memory", what); }

int tcbnn_uploader_create(size_t bytes, int staged, tcbnn_uploader** out) {
    if (out == nullptr) return fail(TCBNN_ENULL, "NULL pointer: out");
    *out = nullptr;
    if (bytes == 0) return fail(TCBNN_EINVAL, "uploader: nothing to upload");
    std::unique_ptr<tcbnn_uploader> u(new (std::nothrow) tcbnn_uploader);
    if (!u) return out_of_memory("uploader");
    u->bytes = bytes;
    u->pinned_bytes = std::min(kPinnedMost, (bytes + kPiece - 1) / kPiece * kPiece);
    int rc = check_hip(hipHostMalloc(&u->pinned, u->pinned_bytes, hipHostMallocDefault), "hipHostMalloc");
    if (rc == TCBNN_OK && staged && bytes >= kOverlapFrom) rc = check_hip(hipMalloc(&u->device, bytes), "hipMalloc");
    if (rc != TCBNN_OK) {
        (void)hipGetLastError();  // (a caller without an uploader copies as it is: the next launch is not to report this)
        return rc;
    }
    if (bytes > 4 * kPiece) {
        try {
            u->workers = Workers::get();
        } catch (const std::exception&) {  // (no memory for them: the caller's own thread does the work)
        }
    }
    *out = u.release();
    return TCBNN_OK;
}

void tcbnn_uploader_destroy(tcbnn_uploader* u) {
    delete u;
}

int tcbnn_upload(tcbnn_uploader* u, void* dst, const void* src_host, size_t bytes) {
    if (u == nullptr || dst == nullptr || src_host == nullptr) return fail(TCBNN_ENULL, "NULL pointer: upload");
    if (bytes > u->bytes) return fail(TCBNN_EINVAL, "upload: longer than the uploader was made for");
    std::lock_guard<std::mutex> l(u->m);
    u->staged = 0;
    try {
        return pass(u, dst, src_host, bytes, nullptr);
    } catch (const std::bad_alloc&) {
        return out_of_memory("upload");
    }
}

int tcbnn_upload_stage(tcbnn_uploader* u, const float* src_host, size_t count, float* abs_max) {
    if (u == nullptr || src_host == nullptr || abs_max == nullptr) return fail(TCBNN_ENULL, "NULL pointer: upload_stage");
    const size_t bytes = 4 * count;
    if (bytes > u->bytes || (u->device == nullptr && bytes > u->pinned_bytes))
        return fail(TCBNN_EINVAL, "upload_stage: longer than the uploader was made for");
    std::lock_guard<std::mutex> l(u->m);
    u->staged = 0;  // (what was staged before is overwritten from here on, whether this call succeeds or not)
    u->on_device = u->device != nullptr;
    uint32_t most = 0;
    try {
        if (int rc = pass(u, u->device, src_host, bytes, &most)) return rc;
    } catch (const std::bad_alloc&) {
        return out_of_memory("upload_stage");
    }
    u->staged = bytes;
    *abs_max = magnitude(most);
    return TCBNN_OK;
}

int tcbnn_upload_commit(tcbnn_uploader* u, void* dst) {
    if (u == nullptr || dst == nullptr) return fail(TCBNN_ENULL, "NULL pointer: upload_commit");
    std::lock_guard<std::mutex> l(u->m);
    if (u->staged == 0) return fail(TCBNN_EINVAL, "upload_commit: nothing is staged");
    const size_t bytes = u->staged;
    u->staged = 0;
    if (int rc = check_hip(hipMemcpyAsync(dst, u->on_device ? u->device : u->pinned, bytes,
                                          u->on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, nullptr),
                           "hipMemcpyAsync"))
        return rc;
    return check_hip(hipStreamSynchronize(nullptr), "hipStreamSynchronize");
}

// max |x| over a host array, on a few host threads (NaN or infinity anywhere: +infinity)
float tcbnn_host_abs_max(const float* values_host, size_t count) {
    if (values_host == nullptr || count == 0) return 0.0f;
    std::atomic<size_t> next{0};
    std::atomic<uint32_t> most{0};
    constexpr size_t kFloats = kPiece / 4;
    auto work = [&] {
        uint32_t m = 0;
        for (;;) {
            const size_t at = next.fetch_add(kFloats, std::memory_order_relaxed);
            if (at >= count) break;
            m = std::max(m, copy_max(nullptr, reinterpret_cast<const uint32_t*>(values_host) + at, std::min(kFloats, count - at), false));
        }
        uint32_t seen = most.load(std::memory_order_relaxed);
        while (m > seen && !most.compare_exchange_weak(seen, m, std::memory_order_relaxed)) {
        }
    };
    const size_t n = std::min<size_t>(std::min<size_t>(count >> 20, 8), std::thread::hardware_concurrency());
    std::vector<std::thread> helpers = start_threads((int)n - 1, work);
    work();
    for (std::thread& t : helpers) t.join();
    return magnitude(most.load());
}

}  // extern "C"
