// afd_xfer.hip -- staged host <-> device copies (host code only).
//
// The runtime's copies between pageable memory and the device reach 38 GB/s up at 12 MB, but on a
// 1.3 GB state 29 GB/s up and 10 GB/s down (one thread takes every page fault of the fresh array the
// state goes to), against 57 GB/s of pinned copies.  Here up to XFER_THREADS threads each take chunks in turn: a DMA between the device and one of the thread's two
// pinned buffers on the caller's stream, and a memcpy between that buffer and the user's array, so that
// the page faults and copies of one thread overlap the DMA of the others.  The 1.3 GB state: up
// 44 -> 28 ms, down 130 -> 29 ms; 45 MB: up 1.60 -> 1.15 ms, down 4.85 -> 1.5 ms.  (4 MB chunks: with 2 MB
// ones the 1.3 GB took 32 ms each way, with 1 MB 41 ms; 12 threads gained nothing over 8.)
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <utility>
#include <vector>

#include <unistd.h>

#include "afd_xfer.hpp"

namespace afd {

namespace {

constexpr int XFER_THREADS = 8;
constexpr size_t CHUNK_MAX = size_t(4) << 20;
constexpr size_t STAGE_BYTES = 2 * CHUNK_MAX * XFER_THREADS;
// Smaller arrays are left to the runtime, which beats the chunks there (24 MB up 0.66 against 0.72 ms,
// 5.6 MB down 0.345 against 0.357; 45 MB up 1.60 against 1.15, 8.6 MB down 0.52 against 0.41)
constexpr size_t UP_MIN = size_t(32) << 20, DOWN_MIN = size_t(7) << 20;

struct Job {
    bool down;
    char *host, *dev;
    size_t bytes, chunk;
    int device;
    hipStream_t stream;
    std::atomic<size_t> next{0};
    std::atomic<int> err{hipSuccess};
};

// The chunks one thread takes of a job, through its two pinned buffers at `stage` and their events.
void work(Job &j, char *stage, hipEvent_t *ev) {
    size_t off[2] = {0, 0}, len[2] = {0, 0};  // len > 0: a DMA of this buffer is in flight
    hipError_t e = hipSetDevice(j.device);
    // ends the DMA of buffer b; downwards the user's array then takes it
    auto finish = [&](int b) {
        if (len[b] == 0) return;
        hipError_t w = hipEventSynchronize(ev[b]);
        if (w == hipSuccess && j.down) memcpy(j.host + off[b], stage + b * CHUNK_MAX, len[b]);
        if (w != hipSuccess && e == hipSuccess) e = w;
        len[b] = 0;
    };
    int b = 0;
    while (e == hipSuccess && j.err.load(std::memory_order_relaxed) == hipSuccess) {
        const size_t o = j.next.fetch_add(1, std::memory_order_relaxed) * j.chunk;
        if (o >= j.bytes) break;
        const size_t n = j.bytes - o < j.chunk ? j.bytes - o : j.chunk;
        finish(b);
        if (e != hipSuccess) break;
        char *buf = stage + b * CHUNK_MAX;
        if (!j.down) memcpy(buf, j.host + o, n);
        e = j.down ? hipMemcpyAsync(buf, j.dev + o, n, hipMemcpyDeviceToHost, j.stream)
                   : hipMemcpyAsync(j.dev + o, buf, n, hipMemcpyHostToDevice, j.stream);
        if (e == hipSuccess) {
            off[b] = o;
            len[b] = n;
            e = hipEventRecord(ev[b], j.stream);
        }
        b ^= 1;
        if (j.down) finish(b);  // the older one, while the newer one's DMA runs
    }
    finish(b);
    finish(b ^ 1);
    if (e != hipSuccess) {
        int none = hipSuccess;
        j.err.compare_exchange_strong(none, (int)e);
        (void)hipStreamSynchronize(j.stream);  // no DMA into the buffers after an error either
    }
}

// The shared staging memory and helper threads.  A copy leases it whole; a copy that finds it leased
// (another thread's) goes through the runtime's own path.  The caller works too and never waits for a
// helper that has not begun, so that a helper that cannot run (a forked child has none) only costs speed.
struct Pool {
    std::mutex lease;  // held for the length of a copy
    std::mutex mu;     // the fields below
    std::condition_variable wake, idle;
    char *stage = nullptr;
    hipEvent_t ev[XFER_THREADS][2] = {};
    int ev_device = -1;
    std::vector<std::thread> helpers;
    Job *job = nullptr;
    unsigned long gen = 0;
    int active = 0;
    bool quit = false;
    const pid_t pid = getpid();

    void helper(int t) {
        unsigned long seen = 0;
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            wake.wait(l, [&] { return quit || (job && gen != seen); });
            if (quit) return;
            seen = gen;
            Job *j = job;
            ++active;
            l.unlock();
            work(*j, stage + (size_t)t * 2 * CHUNK_MAX, ev[t]);
            l.lock();
            if (--active == 0) idle.notify_all();
        }
    }

    void drop_events() {
        for (auto &pair : ev)
            for (hipEvent_t &x : pair) {
                if (x) (void)hipEventDestroy(x);
                x = nullptr;
            }
        ev_device = -1;
    }

    // With the lease held: the staging memory, the helpers and the events of `device`.
    bool start(int device) {
        if (ev_device != device) {
            drop_events();
            for (auto &pair : ev)
                for (hipEvent_t &x : pair)
                    if (hipEventCreateWithFlags(&x, hipEventDisableTiming) != hipSuccess) {
                        (void)hipGetLastError();
                        x = nullptr;
                        drop_events();
                        return false;
                    }
            ev_device = device;
        }
        if (stage) return true;
        void *p = nullptr;
        if (hipHostMalloc(&p, STAGE_BYTES, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        stage = (char *)p;
        const int hw = (int)std::thread::hardware_concurrency();
        const int n = hw >= 2 * XFER_THREADS ? XFER_THREADS : (hw / 2 > 1 ? hw / 2 : 1);
        try {
            for (int t = 1; t < n; ++t) helpers.emplace_back([this, t] { helper(t); });
        } catch (...) {  // fewer threads: slower, still whole
        }
        return true;
    }

    void run(Job &j) {  // with the lease held
        {
            std::lock_guard<std::mutex> l(mu);
            job = &j;
            ++gen;
        }
        // a helper pays from about two chunks of its own on
        const size_t chunks = (j.bytes + j.chunk - 1) / j.chunk;
        for (size_t k = 0; k < helpers.size() && 2 * (k + 1) < chunks; ++k) wake.notify_one();
        work(j, stage, ev[0]);
        std::unique_lock<std::mutex> l(mu);
        job = nullptr;  // a helper that wakes from here on finds nothing to begin
        idle.wait(l, [&] { return active == 0; });
    }

    ~Pool() {
        {
            std::lock_guard<std::mutex> l(mu);
            quit = true;
        }
        wake.notify_all();
        for (auto &t : helpers) t.join();
        drop_events();
        if (stage) (void)hipHostFree(stage);
    }
};

std::mutex g_mu;
int g_refs = 0;
char *g_pins[2] = {};    // free pinned blocks
Pool *g_pool = nullptr;  // never a static object: a process that exits with contexts open must not join

hipError_t copy(bool down, void *host, void *dev, size_t bytes, hipStream_t s, bool wait) {
    auto direct = [&]() {
        hipError_t e = down ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s)
                            : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
        return e == hipSuccess && wait ? hipStreamSynchronize(s) : e;
    };
    if (bytes < (down ? DOWN_MIN : UP_MIN)) return direct();
    Pool *p;
    {
        std::lock_guard<std::mutex> l(g_mu);
        if (!g_pool) g_pool = new (std::nothrow) Pool;
        p = g_pool;
    }
    if (!p) return direct();
    std::unique_lock<std::mutex> lease(p->lease, std::try_to_lock);
    Job j;
    hipError_t e = hipGetDevice(&j.device);
    if (e != hipSuccess) return e;
    if (!lease.owns_lock() || !p->start(j.device)) return direct();
    j.down = down;
    j.host = (char *)host;
    j.dev = (char *)dev;
    j.bytes = bytes;
    size_t c = bytes / (2 * XFER_THREADS);  // two chunks a thread, whole pages
    c = c > CHUNK_MAX ? CHUNK_MAX : c;
    j.chunk = (c + 4095) & ~size_t(4095);
    j.stream = s;
    p->run(j);
    return (hipError_t)j.err.load();
}

}  // namespace

void xfer_retain() {
    std::lock_guard<std::mutex> l(g_mu);
    ++g_refs;
}

char *xfer_pin_get(bool lock) {
    {
        std::lock_guard<std::mutex> l(g_mu);
        for (char *&b : g_pins)
            if (b) {
                char *r = b;
                b = nullptr;
                return r;
            }
    }
    if (!lock) return nullptr;
    void *p = nullptr;
    if (hipHostMalloc(&p, PIN_BLOCK, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return (char *)p;
}

void xfer_pin_put(char *block) {
    {
        std::lock_guard<std::mutex> l(g_mu);
        for (char *&b : g_pins)
            if (!b) {
                b = block;
                return;
            }
    }
    (void)hipHostFree(block);
}

void xfer_release() {
    Pool *p = nullptr;
    char *pins[2] = {};
    {
        std::lock_guard<std::mutex> l(g_mu);
        if (--g_refs == 0) {
            p = g_pool;
            g_pool = nullptr;
            std::swap(pins[0], g_pins[0]);
            std::swap(pins[1], g_pins[1]);
        }
    }
    for (char *b : pins)
        if (b) (void)hipHostFree(b);
    if (p && p->pid == getpid()) delete p;  // a forked child has no threads to join
}

hipError_t xfer_d2h(void *host, const void *dev, size_t bytes, hipStream_t s, bool wait) {
    return copy(true, host, (void *)dev, bytes, s, wait);
}
hipError_t xfer_h2d(void *dev, const void *host, size_t bytes, hipStream_t s, bool wait) {
    return copy(false, (void *)host, dev, bytes, s, wait);
}

}  // namespace afd
