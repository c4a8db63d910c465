// download.hip -- device arrays to the caller's (pageable) host memory.
//
// A plain copy into pageable memory takes the page faults of a fresh array on one
// thread: 4.4 GB/s, 123 ms for the four fields of 256^3 (as much as 200 FP64
// steps); into an array in use, 17 GB/s.  Large downloads go through pinned staging
// instead: the device copies a chunk into one slot while the one before is copied
// on into the caller's array.  The calling thread does that by itself at no less
// than the plain copy's rate (measured on MI355X, ms, plain / by itself: 17 MB
// fresh 3.8 / 3.5, in use 0.98 / 0.67; 134 MB 31 / 27 and 7.7 / 5.0; beside 16
// threads that keep all 16 CPUs of the process busy, 17 MB 8.1 / 7.7 and 0.98 /
// 0.70).  Helper threads take chunks beside it (134 MB fresh 10, 537 MB 39), but
// are never waited for unless they hold one: with every CPU busy a new thread first
// runs some 4 ms later, and downloads that waited for their threads took 4.0 ms
// for 17 and 34 MB in use where the plain copy takes 1.0 and 2.0 (so: 0.9, 1.3).
#include <hip/hip_runtime.h>
#include <sched.h>

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "context.hpp"

namespace {

// Bytes of a staging slot.  A copy command costs the device 15 us, after an idle time
// over 100 until its clocks are up: 134 MB in chunks of 512 KiB took 6.4 and 30 ms, of
// 1 MiB 4.4 and 20, of 2 MiB 3.5 and 11.5 (plain 7.7 and 20).
constexpr size_t CHUNK = 2u << 20;
constexpr int WORKERS = 4, SLOTS = 2;      // 16 MiB of pinned memory
// Smaller downloads: the plain copy (65^3, 8.8 MB: 2.1 ms fresh, 0.5 in use).  The
// first download also pins the slots and takes their page faults, 0.4 ms per MiB,
// which from here on the faults saved pay for (17 MB into a fresh array from a
// fresh context: 4.3 ms plain, 2.3).
constexpr size_t STAGED_FROM = 16u << 20;

// The staging memory, one for the process: taken on the first large download, used
// by one download at a time (another goes the plain way) and given back with the
// last context.
std::mutex g_mu;
std::condition_variable g_cv;  // g_helpers fell
char* g_staging = nullptr;
bool g_in_use = false;
int g_users = 0;
int g_helpers = 0;  // helper threads not at their end yet

char* take_staging() {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_in_use) return nullptr;
    if (!g_staging && hipHostMalloc(reinterpret_cast<void**>(&g_staging), CHUNK * WORKERS * SLOTS,
                                    hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        g_staging = nullptr;
        return nullptr;
    }
    g_in_use = true;
    return g_staging;
}

void give_back_locked() {
    if (g_users == 0 && !g_in_use && g_staging) {
        (void)hipHostFree(g_staging);
        g_staging = nullptr;
    }
}

struct Chunk {
    char* dst;
    const char* src;
    size_t bytes;
};

// One download: its chunks, who takes the next, and how many are still to come.
// Helpers hold it too, so that one that starts after the end finds nothing left.
struct Job {
    int device;
    hipStream_t stream;
    std::vector<Chunk> chunks;
    std::atomic<size_t> next{0};
    std::atomic<int> err{hipSuccess};  // the first error; the rest of the chunks is then only counted
    std::mutex mu;
    std::condition_variable cv;
    size_t left = 0;

    void done(size_t n) {
        std::lock_guard<std::mutex> lock(mu);
        if ((left -= n) == 0) cv.notify_all();
    }
    void failed(hipError_t e) {
        int none = hipSuccess;
        err.compare_exchange_strong(none, (int)e);
    }
};

// Takes chunks through `slots` until none is left.
void work(Job& job, char* slots, unsigned event_flags) {
    size_t c = job.next.fetch_add(1);
    if (c >= job.chunks.size()) return;  // (nothing of the job is touched after its end)
    int caller = job.device;  // the calling thread keeps its own device
    (void)hipGetDevice(&caller);
    hipEvent_t ready[SLOTS] = {};
    hipError_t e = hipSetDevice(job.device);
    for (auto& ev : ready)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, event_flags | hipEventDisableTiming);
    if (e != hipSuccess) job.failed(e);
    const Chunk* held[SLOTS] = {};
    size_t finished = 0;  // told to the job at the end: a helper keeps its slots till then
    for (int at = 0, full = 0; c < job.chunks.size() || full > 0; at = (at + 1) % SLOTS) {
        char* slot = slots + at * CHUNK;
        if (held[at]) {
            e = hipEventSynchronize(ready[at]);
            if (e == hipSuccess) std::memcpy(held[at]->dst, slot, held[at]->bytes);
            else job.failed(e);
            held[at] = nullptr;
            --full;
            ++finished;
        }
        if (c >= job.chunks.size()) continue;
        if (job.err.load() == hipSuccess) {
            const Chunk& k = job.chunks[c];
            e = hipMemcpyAsync(slot, k.src, k.bytes, hipMemcpyDeviceToHost, job.stream);
            if (e == hipSuccess) e = hipEventRecord(ready[at], job.stream);
            if (e == hipSuccess) {
                held[at] = &k;
                ++full;
            } else {
                job.failed(e);
                (void)hipStreamSynchronize(job.stream);  // no copy into the slot is left
                ++finished;
            }
        } else {
            ++finished;
        }
        c = job.next.fetch_add(1);
    }
    for (hipEvent_t ev : ready)
        if (ev) (void)hipEventDestroy(ev);
    if (caller != job.device) (void)hipSetDevice(caller);
    job.done(finished);
}

// Memory a device copy can write directly (pinned, managed, a device's).
bool known_to_device(const void* p) {
    hipPointerAttribute_t a{};
    const bool known = hipPointerGetAttributes(&a, p) == hipSuccess && a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return known;
}

int host_threads() {
    cpu_set_t set;
    CPU_ZERO(&set);
    const int n = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    return n < WORKERS ? n : WORKERS;
}

void start_helper(const std::shared_ptr<Job>& job, char* slots) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        ++g_helpers;
    }
    auto over = [] {
        std::lock_guard<std::mutex> lock(g_mu);
        --g_helpers;
        g_cv.notify_all();
    };
    try {
        // (a blocked wait, not a spinning one: the CPU is the other threads')
        std::thread([job, slots, over] {
            work(*job, slots, hipEventBlockingSync);
            over();
        }).detach();
    } catch (...) {  // fewer threads, then
        over();
    }
}

// All chunks through the staging memory; false where that cannot be had.
bool staged(int device, hipStream_t stream, const lbm_copy* copies, int count, hipError_t* err) {
    std::shared_ptr<Job> job;
    try {
        job = std::make_shared<Job>();
        for (int q = 0; q < count; ++q)
            for (size_t o = 0; copies[q].dst && o < copies[q].bytes; o += CHUNK)
                job->chunks.push_back({static_cast<char*>(copies[q].dst) + o, static_cast<const char*>(copies[q].src) + o,
                                       copies[q].bytes - o < CHUNK ? copies[q].bytes - o : CHUNK});
    } catch (...) {  // no memory for the list of chunks
        return false;
    }
    char* slots = take_staging();
    if (!slots) return false;
    job->device = device;
    job->stream = stream;
    job->left = job->chunks.size();
    *err = hipStreamSynchronize(stream);  // one thread waits for the work before, not all of them
    if (*err == hipSuccess) {
        const int n = host_threads();
        for (int t = 1; t < n; ++t) start_helper(job, slots + t * SLOTS * CHUNK);
        work(*job, slots, hipEventDefault);
        std::unique_lock<std::mutex> lock(job->mu);
        job->cv.wait(lock, [&] { return job->left == 0; });
        *err = (hipError_t)job->err.load();
    }
    std::lock_guard<std::mutex> lock(g_mu);
    g_in_use = false;
    give_back_locked();
    return true;
}

}  // namespace

void lbm_staging_user(int change) {
    std::unique_lock<std::mutex> lock(g_mu);
    g_users += change;
    give_back_locked();
    if (g_users == 0) g_cv.wait(lock, [] { return g_helpers == 0; });  // none is left in the library
}

int lbm_download(int device, hipStream_t stream, const lbm_copy* copies, int count) {
    size_t total = 0;
    bool pageable = true;
    for (int q = 0; q < count; ++q) {
        if (!copies[q].dst) continue;
        total += copies[q].bytes;
        if (copies[q].bytes && known_to_device(copies[q].dst)) pageable = false;
    }
    hipError_t e = hipSuccess;
    if (total >= STAGED_FROM && pageable && staged(device, stream, copies, count, &e)) {
        if (e != hipSuccess) return lbm_fail(LBM_ERR_HIP, "download failed: %s", hipGetErrorString(e));
        return LBM_OK;
    }
    for (int q = 0; q < count; ++q)
        if (copies[q].dst)
            HIP_TRY(hipMemcpyAsync(copies[q].dst, copies[q].src, copies[q].bytes, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return LBM_OK;
}
