// download.hip -- device arrays to the caller's (pageable) host memory.
//
// A plain copy into pageable memory runs on one host thread, which also takes
// the page faults of a fresh array: 10 GB/s for the fields of 256^3 (52 ms, as
// much as 57 FP64 steps).  Large downloads go through pinned staging instead:
// a few threads each bring chunks into their own two pinned slots (the device
// copies the next while the thread empties the last into the caller's array).
// Measured on MI355X, 256^3, four fields into a fresh array: 52 -> 14.4 ms with
// four threads (eight: 14.1).
#include <hip/hip_runtime.h>
#include <sched.h>

#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "context.hpp"

namespace {

constexpr size_t CHUNK = 2u << 20;         // bytes of a staging slot
constexpr int WORKERS = 4, SLOTS = 2;      // 16 MiB of pinned memory
constexpr size_t STAGED_FROM = 16u << 20;  // smaller downloads: the plain copy (65^3: 0.55 ms either way)

// The staging memory, one for the process: pinning it takes some ms, which
// every context would pay on its first output.  It is taken on the first large
// download, used by one download at a time (another goes the plain way) and
// given back with the last context.
std::mutex g_mu;
char* g_staging = nullptr;
bool g_in_use = false;
int g_users = 0;

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

// Chunks next, next + 1, ... through two pinned slots.  Stops at the first
// error, which it returns.
hipError_t work(int device, hipStream_t stream, const std::vector<Chunk>& chunks, std::atomic<size_t>& next,
                char* slots) {
    int caller = device;  // the calling thread takes part and keeps its own device
    (void)hipGetDevice(&caller);
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return e;
    hipEvent_t done[SLOTS] = {};
    for (auto& ev : done)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    size_t held[SLOTS];
    bool full[SLOTS] = {};
    int at = 0;
    for (bool more = true; e == hipSuccess;) {
        const size_t c = more ? next.fetch_add(1) : chunks.size();
        more = c < chunks.size();
        if (!more && !full[0] && !full[1]) break;
        if (more) {
            e = hipMemcpyAsync(slots + at * CHUNK, chunks[c].src, chunks[c].bytes, hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(done[at], stream);
            held[at] = c;
            full[at] = e == hipSuccess;
        }
        at = 1 - at;  // the slot filled the turn before
        if (full[at]) {
            const hipError_t w = hipEventSynchronize(done[at]);
            if (e == hipSuccess) e = w;
            if (e == hipSuccess) std::memcpy(chunks[held[at]].dst, slots + at * CHUNK, chunks[held[at]].bytes);
            full[at] = false;
        }
    }
    for (int s = 0; s < SLOTS; ++s) {
        if (full[s]) (void)hipEventSynchronize(done[s]);  // after an error: no copy into the slot is left
        if (done[s]) (void)hipEventDestroy(done[s]);
    }
    if (caller != device) (void)hipSetDevice(caller);
    return e;
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

// All chunks through the staging memory; false where that cannot be had.
bool staged(int device, hipStream_t stream, const lbm_copy* copies, int count, hipError_t* err) {
    char* slots = take_staging();
    if (!slots) return false;
    // One thread waits for the work before, not all of them: waiting spins, and with
    // a caller's own host threads at work it went over the process's CPU share
    // (128^3 FP16 in two subdomains, 33 MB each, converted by 16 threads after the
    // copy: 12 to 48 ms a pass with four waiting, 12.0 with one).
    *err = hipStreamSynchronize(stream);
    bool ran = *err != hipSuccess;
    if (!ran) try {
        std::vector<Chunk> chunks;
        for (int q = 0; q < count; ++q)
            for (size_t o = 0; copies[q].dst && o < copies[q].bytes; o += CHUNK)
                chunks.push_back({static_cast<char*>(copies[q].dst) + o, static_cast<const char*>(copies[q].src) + o,
                                  copies[q].bytes - o < CHUNK ? copies[q].bytes - o : CHUNK});
        std::atomic<size_t> next{0};
        hipError_t e[WORKERS] = {};
        std::vector<std::thread> threads;
        const int n = host_threads();
        threads.reserve(n);
        try {
            for (int t = 1; t < n; ++t)
                threads.emplace_back([&, t] { e[t] = work(device, stream, chunks, next, slots + t * SLOTS * CHUNK); });
        } catch (...) {  // fewer threads, then
        }
        e[0] = work(device, stream, chunks, next, slots);
        for (auto& t : threads) t.join();
        *err = hipSuccess;
        for (hipError_t x : e)
            if (x != hipSuccess) *err = x;
        ran = true;
    } catch (...) {  // no memory for the list of chunks: nothing was started
    }
    std::lock_guard<std::mutex> lock(g_mu);
    g_in_use = false;
    give_back_locked();
    return ran;
}

}  // namespace

void lbm_staging_user(int change) {
    std::lock_guard<std::mutex> lock(g_mu);
    g_users += change;
    give_back_locked();
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
