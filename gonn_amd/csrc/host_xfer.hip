// host_xfer.hip -- transfers of the fp64 host entry points.
//
// The arrays are pageable host memory. A copy straight from or to it goes
// through the runtime's own staging on one thread, moves fp64 over the bus
// where the kernels take fp32, and a download into memory that was never
// touched (a caller's fresh result array) takes its page faults on that thread
// too: 16.8 MB arrays measured 30 GB/s up and 4 GB/s down. Here up to
// kThreads threads each convert (or copy) chunks between the arrays and two
// pinned slots of their own, so conversion, page faults and the bus overlap:
// eight such arrays up 4.9 -> 2.3 ms, four down 15.9 -> 2.8 ms, and a training
// call pair at BH 32, S 1024, d 64 17.6 -> 6.9 ms. Small calls use fewer
// threads, down to the calling one.
#include "host_xfer.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace gonn {

namespace {

constexpr int kThreads = 8;
constexpr size_t kSlot = (size_t)1 << 20;  // bytes of a pinned slot (256 KB chunks: half the rate)
constexpr size_t kLane = 2 * kSlot;        // what one thread works with

// Pinned lanes, one per thread of a transfer in flight. At most kMaxLanes exist
// (64 MB), each made when a transfer first needs it; those that stayed unused
// over kWindow transfers are freed. A transfer that finds none left stages
// through ordinary memory.
constexpr int kMaxLanes = 4 * kThreads, kWindow = 64;
std::mutex g_mu;
void* g_free[kMaxLanes];
int g_nfree = 0, g_made = 0;
int g_idle = 0, g_count = 0;  // least g_nfree since, and transfers in, this window

struct Staging {
    void* lane[kThreads];
    int n = 0;
    explicit Staging(int want) {
        int make = 0;
        {
            std::lock_guard<std::mutex> lock(g_mu);
            while (n < want && g_nfree > 0) lane[n++] = g_free[--g_nfree];
            g_idle = std::min(g_idle, g_nfree);
            make = std::min(want - n, kMaxLanes - g_made);
            g_made += make;
        }
        for (; make > 0; make--) {
            if (hipHostMalloc(&lane[n], kLane, hipHostMallocPortable) != hipSuccess) {
                (void)hipGetLastError();
                std::lock_guard<std::mutex> lock(g_mu);
                g_made -= make;
                break;
            }
            n++;
        }
    }
    ~Staging() {
        void* drop[kMaxLanes];
        int nd = 0;
        {
            std::lock_guard<std::mutex> lock(g_mu);
            for (int i = 0; i < n; i++) g_free[g_nfree++] = lane[i];
            if (++g_count == kWindow) {
                while (nd < g_idle) drop[nd++] = g_free[--g_nfree];
                g_made -= nd;
                g_count = 0;
                g_idle = g_nfree;
            }
        }
        for (int i = 0; i < nd; i++)
            if (hipHostFree(drop[i]) != hipSuccess) (void)hipGetLastError();
    }
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
};

size_t row_bytes(const HostCopy& c) { return c.dp ? (size_t)c.dp * 4 : (size_t)c.d * 8; }

// Rows [r0, r0 + n) between the host array and a staged chunk.
void pack(const HostCopy& c, size_t r0, size_t n, void* chunk) {
    const double* src = c.host + r0 * c.d;
    if (!c.dp) {
        std::memcpy(chunk, src, n * c.d * 8);
        return;
    }
    float* dst = (float*)chunk;
    if (c.dp == c.d) {
        for (size_t i = 0; i < n * c.d; i++) dst[i] = (float)src[i];
        return;
    }
    for (size_t r = 0; r < n; r++, src += c.d, dst += c.dp) {
        for (int i = 0; i < c.d; i++) dst[i] = (float)src[i];
        for (int i = c.d; i < c.dp; i++) dst[i] = 0.f;
    }
}
void unpack(const HostCopy& c, size_t r0, size_t n, const void* chunk) {
    double* dst = c.host + r0 * c.d;
    if (!c.dp) {
        std::memcpy(dst, chunk, n * c.d * 8);
        return;
    }
    const float* src = (const float*)chunk;
    if (c.dp == c.d) {
        for (size_t i = 0; i < n * c.d; i++) dst[i] = (double)src[i];
        return;
    }
    for (size_t r = 0; r < n; r++, dst += c.d, src += c.dp)
        for (int i = 0; i < c.d; i++) dst[i] = (double)src[i];
}

struct Chunk {
    const HostCopy* c;
    size_t r0, n;
};

// One thread's share: chunks from `next` on, through its two slots. Every
// copy that uses a slot has finished when this returns.
hipError_t run_share(const std::vector<Chunk>& chunks, std::atomic<size_t>& next, bool up, int dev,
                     char* slots, bool pinned, hipStream_t s) {
    hipError_t e = hipSetDevice(dev);
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (int i = 0; i < 2 && e == hipSuccess; i++)
        e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    const Chunk* busy[2] = {nullptr, nullptr};
    // Waits for slot i's copy; a download's chunk then goes to the host array.
    auto finish = [&](int i) {
        if (!busy[i]) return;
        const hipError_t w = pinned ? hipEventSynchronize(ev[i]) : hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        if (!up && e == hipSuccess) unpack(*busy[i]->c, busy[i]->r0, busy[i]->n, slots + i * kSlot);
        busy[i] = nullptr;
    };
    for (int i = 0; e == hipSuccess; i ^= 1) {
        const size_t j = next.fetch_add(1, std::memory_order_relaxed);
        if (j >= chunks.size()) break;
        const Chunk& k = chunks[j];
        char* slot = slots + i * kSlot;
        char* d = (char*)k.c->dev + k.r0 * row_bytes(*k.c);
        const size_t bytes = k.n * row_bytes(*k.c);
        if (up) {
            finish(i);
            if (e != hipSuccess) break;
            pack(*k.c, k.r0, k.n, slot);
            e = hipMemcpyAsync(d, slot, bytes, hipMemcpyHostToDevice, s);
        } else {
            e = hipMemcpyAsync(slot, d, bytes, hipMemcpyDeviceToHost, s);
        }
        if (e != hipSuccess) break;
        busy[i] = &k;
        e = hipEventRecord(ev[i], s);
        if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no event to wait for
        if (!up) finish(i ^ 1);  // while this chunk's copy runs
    }
    finish(0);
    finish(1);
    for (hipEvent_t x : ev)
        if (x) (void)hipEventDestroy(x);
    return e;
}

hipError_t transfer(const HostCopy* c, int n, bool up, hipStream_t s) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    try {
        std::vector<Chunk> chunks;
        size_t total = 0;
        for (int i = 0; i < n; i++) {
            const size_t rb = row_bytes(c[i]), per = std::max<size_t>(1, kSlot / rb);
            for (size_t r = 0; r < c[i].rows; r += per)
                chunks.push_back({&c[i], r, std::min(per, c[i].rows - r)});
            total += c[i].rows * rb;
        }
        const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
        int nt = (int)std::min<size_t>({(size_t)kThreads, (size_t)hw, 1 + total / kLane,
                                        std::max<size_t>(1, chunks.size())});
        Staging st(nt);
        const bool pinned = st.n > 0;
        if (pinned) nt = st.n;
        std::vector<char> heap(pinned ? 0 : (size_t)nt * kLane);
        auto slots = [&](int k) { return pinned ? (char*)st.lane[k] : heap.data() + k * kLane; };
        std::atomic<size_t> next{0};
        std::vector<hipError_t> err(nt, hipSuccess);
        std::vector<std::thread> th;
        th.reserve(nt);
        for (int k = 1; k < nt; k++) {
            try {
                th.emplace_back([&, k] {
                    err[k] = run_share(chunks, next, up, dev, slots(k), pinned, s);
                });
            } catch (const std::exception&) {
                break;  // no thread (or memory for one) to be had: the others take its chunks
            }
        }
        err[0] = run_share(chunks, next, up, dev, slots(0), pinned, s);
        for (std::thread& t : th) t.join();
        for (hipError_t x : err)
            if (e == hipSuccess) e = x;
    } catch (const std::bad_alloc&) {
        return hipErrorOutOfMemory;
    }
    return e;
}

}  // namespace

hipError_t host_upload(const HostCopy* c, int n, hipStream_t s) { return transfer(c, n, true, s); }
hipError_t host_download(const HostCopy* c, int n, hipStream_t s) {
    return transfer(c, n, false, s);
}

}  // namespace gonn
