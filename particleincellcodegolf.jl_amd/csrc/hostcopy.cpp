// hostcopy.cpp -- device-to-host copies through pinned staging buffers by
// several host threads.
//
// What bounds a copy into ordinary memory is the host: one thread that fills
// pages the caller has never touched and unpacks the mixed formats moves about
// 2 to 10 GB/s, a fraction of the link.  Here each of up to kWorkers threads
// has a slab of two pinned buffers; it takes the next chunk of the list, starts
// its transfer into one buffer, and meanwhile unpacks the other into the
// caller's array.  168 MB of doubles (2 MiB pages / 4 KiB pages): one thread
// 15.6 / 42 ms, two 6.7 / 24, four 4.8 / 13, eight 5.0 / 8.  On a host whose
// cores are all busy with others' work: one 48 / 84, eight 12 / 25.
//
// A list of at most a slab is one kernel that converts and writes it into
// pinned memory over the link, and one wait: an array at a time, each of its
// transfers and waits costs 20-30 us, and starting the threads 0.2 ms.  A single
// array of doubles has nothing to save there and goes straight into the
// caller's memory (32 KB: 11.5 us, and 15.9 through the kernel; 800 KB: 58 both
// ways).
//
// A worker to every chunk; but a device's first two such copies make no more
// slabs than one to every 4 MiB of theirs, and a second stream only for more than
// two: making and freeing them costs some 0.1 ms each, which a program with a
// context to a run, and a copy or two from it, would pay every time (4e5 FP64
// particles, 6.4 MB, from create to destroy: 2.0 ms, with all at once 4.0, in
// pageable memory 2.2).  A program that goes on reading gets them all (a grid of
// 4 MiB in 0.30 ms; 0.65 by two, 0.69 in pageable memory).
//
// A copy takes the slabs that are free and never waits for another's: where
// there is none (or no pinned memory to make one), it goes through pageable
// memory on the caller's stream.
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace pic {

namespace {

constexpr int kWorkers = 8;                      // slabs one copy takes at most
constexpr int kSlabs = 2 * kWorkers;             // slabs of a device, made when they are needed
constexpr size_t kChunkBytes = size_t(1) << 20;  // of one pinned buffer
constexpr size_t kSlabBytes = 2 * kChunkBytes;
constexpr int kFirst = 2;                        // copies that make few slabs

struct Slab {
    char* pin = nullptr;  // two buffers
    hipEvent_t done[2] = {nullptr, nullptr};
};

void free_slab(Slab& s) {
    for (hipEvent_t e : s.done)
        if (e) (void)hipEventDestroy(e);
    if (s.pin) (void)hipHostFree(s.pin);
    s = Slab();
}

bool make_slab(Slab& s) {
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&s.pin), kSlabBytes, hipHostMallocDefault);
    if (e != hipSuccess) s.pin = nullptr;
    // waited for by spinning: a sleeping thread wakes too late for a copy of a
    // chunk or two (4 MiB by four: 0.30 ms, asleep 0.45 to 0.63)
    for (hipEvent_t& d : s.done)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&d, hipEventDisableTiming);
    if (e == hipSuccess) return true;
    free_slab(s);
    (void)hipGetLastError();
    return false;
}

// A device's slabs.  The lock is held to take and give slabs only.
struct Pool {
    std::mutex m;
    int made = 0;              // slabs that exist, free or taken
    int copies = 0;            // by several workers so far
    Slab idle[kSlabs];         // the free ones
    int nidle = 0;
    // the workers' streams: with one, transfers and the waits for them queue
    // behind each other (168 MB in 8.2 ms against 5.2 with eight); each costs a
    // process 3 ms when it is first made.  A first copy's first one is the caller's.
    hipStream_t own[2] = {nullptr, nullptr};

    void make_stream(hipStream_t& s) {
        if (s || hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess) return;
        s = nullptr;
        (void)hipGetLastError();
    }
    // up to `want` slabs, of which a first copy makes those up to `few`; streams
    // (the caller's, both, on entry): the ones to use in turn
    int take(Slab* out, int want, int few = 1, hipStream_t* streams = nullptr) {
        std::lock_guard<std::mutex> l(m);
        int n = 0;
        while (n < want && nidle > 0) out[n++] = idle[--nidle];
        const bool first = !streams || copies++ < kFirst;
        const int make = first ? few : want;
        for (; n < make && made < kSlabs; ++made)
            if (!make_slab(out[n++])) {
                --n;
                break;
            }
        if (streams && n > (first ? 2 : 1)) make_stream(own[1]);
        if (streams && n > 1 && !first) make_stream(own[0]);
        if (streams && n > 1)
            for (int k = 0; k < 2; ++k)
                if (own[k]) streams[k] = own[k];
        return n;
    }
    void give(const Slab* s, int n) {
        std::lock_guard<std::mutex> l(m);
        for (int k = 0; k < n; ++k) idle[nidle++] = s[k];
    }
    ~Pool() {
        while (nidle > 0) free_slab(idle[--nidle]);
        for (hipStream_t s : own)
            if (s) (void)hipStreamDestroy(s);
    }
};

struct Held {
    std::unique_ptr<Pool> pool;
    int users = 0;
};
std::mutex g_pools_m;
std::map<int, Held>& pools() {
    static std::map<int, Held>* p = new std::map<int, Held>;  // lives as long as any context may
    return *p;
}
Pool* pool_of(int device) {
    std::lock_guard<std::mutex> l(g_pools_m);
    const auto it = pools().find(device);
    return it == pools().end() ? nullptr : it->second.pool.get();
}

size_t element_bytes(CopyKind k) { return k == kCopyF64 || k == kCopyPickF64 ? 8 : 4; }
int sources(CopyKind k) { return k == kCopyPair32 ? 2 : 1; }

struct Chunk {
    const CopyOut* a;
    size_t at, n;
};

// Starts a chunk's transfers into buf, one source behind the other.
hipError_t fetch(const Chunk& c, char* buf, hipStream_t stream) {
    const size_t bytes = element_bytes(c.a->kind) * c.n;
    hipError_t e = hipSuccess;
    for (int k = 0; k < sources(c.a->kind) && e == hipSuccess; ++k)
        e = hipMemcpyAsync(buf + bytes * k, static_cast<const char*>(c.a->src[k]) + element_bytes(c.a->kind) * c.at, bytes,
                           hipMemcpyDeviceToHost, stream);
    return e;
}

void unpack(const Chunk& c, const char* buf) {
    double* o = c.a->dst + c.at;
    const size_t n = c.n;
    switch (c.a->kind) {
    case kCopyF64:
    case kCopyPickF64:
        std::memcpy(o, buf, 8 * n);
        break;
    case kCopyFix32: {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(buf);
        for (size_t j = 0; j < n; ++j) o[j] = (double)q[j] * 0x1p-32;
        break;
    }
    case kCopyUnimod32: {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(buf);
        for (size_t j = 0; j < n; ++j) o[j] = q[j] ? (double)q[j] * 0x1p-32 : 1.0;
        break;
    }
    case kCopyPair32: {
        const float* h = reinterpret_cast<const float*>(buf);
        const float* l = h + n;
        const double s = c.a->scale;
        for (size_t j = 0; j < n; ++j) o[j] = ((double)h[j] + (double)l[j]) * s;
        break;
    }
    }
}

// Chunks off the shared counter until none is left; one transfer ahead.
void work(const Slab& w, hipStream_t stream, int device, const std::vector<Chunk>& chunks, std::atomic<size_t>& next,
          std::atomic<int>& error) {
    auto fail = [&](hipError_t e) {
        int none = hipSuccess;
        error.compare_exchange_strong(none, (int)e);
    };
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return fail(e);
    const Chunk* flying = nullptr;
    for (int s = 0;; s ^= 1) {
        const size_t i = error.load() == hipSuccess ? next.fetch_add(1) : chunks.size();
        const Chunk* c = i < chunks.size() ? &chunks[i] : nullptr;
        if (c) {
            e = fetch(*c, w.pin + s * kChunkBytes, stream);
            if (e == hipSuccess) e = hipEventRecord(w.done[s], stream);
        }
        if (flying && e == hipSuccess) {
            e = hipEventSynchronize(w.done[s ^ 1]);
            if (e == hipSuccess) unpack(*flying, w.pin + (s ^ 1) * kChunkBytes);
        }
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(stream);  // nothing may write the buffers later
            return fail(e);
        }
        if (!c) return;
        flying = c;
    }
}

// Doubles straight into the caller's memory.
hipError_t copy_direct(hipStream_t stream, const CopyOut& a) {
    const hipError_t e = hipMemcpyAsync(a.dst, a.src[0], 8 * a.n, hipMemcpyDeviceToHost, stream);
    const hipError_t done = hipStreamSynchronize(stream);
    return e == hipSuccess ? done : e;
}

// Without a slab: through pageable memory on the caller's stream.
hipError_t copy_plain(hipStream_t stream, const std::vector<Chunk>& chunks, const std::vector<CopyOut>& items) {
    for (const CopyOut& a : items)
        if (element_bytes(a.kind) == 8)
            if (const hipError_t e = copy_direct(stream, a)) return e;
    std::unique_ptr<char, void (*)(void*)> buf(nullptr, std::free);
    for (const Chunk& c : chunks) {
        if (element_bytes(c.a->kind) == 8) continue;
        if (!buf) buf.reset(static_cast<char*>(std::malloc(kChunkBytes)));
        if (!buf) return hipErrorOutOfMemory;
        hipError_t e = fetch(c, buf.get(), stream);
        const hipError_t done = hipStreamSynchronize(stream);
        if (e == hipSuccess) e = done;
        if (e != hipSuccess) return e;
        unpack(c, buf.get());
    }
    return hipSuccess;
}

hipError_t copy_small(const Slab& w, hipStream_t stream, const std::vector<CopyOut>& items) {
    SmallList l{};
    for (const CopyOut& a : items) {
        l.a[l.n] = a;
        l.off[l.n + 1] = l.off[l.n] + a.n;
        ++l.n;
    }
    hipError_t e = launch_copy_small(l, reinterpret_cast<double*>(w.pin), stream);
    const hipError_t done = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = done;
    if (e != hipSuccess) return e;
    for (int k = 0; k < l.n; ++k) std::memcpy(l.a[k].dst, w.pin + 8 * l.off[k], 8 * l.a[k].n);
    return hipSuccess;
}

hipError_t copy_long(const Slab* slabs, int n, int device, const hipStream_t* streams, const std::vector<Chunk>& chunks) {
    std::atomic<size_t> next(0);
    std::atomic<int> error(hipSuccess);
    std::vector<std::thread> threads;
    try {
        for (int k = 1; k < n; ++k)
            threads.emplace_back([&, k] { work(slabs[k], streams[k & 1], device, chunks, next, error); });
    } catch (...) {
        // fewer threads than asked for: the others take their chunks
    }
    work(slabs[0], streams[0], device, chunks, next, error);
    for (std::thread& t : threads) t.join();
    return (hipError_t)error.load();
}

}  // namespace

bool hostcopy_retain(int device) {
    try {
        std::lock_guard<std::mutex> l(g_pools_m);
        Held& h = pools()[device];
        if (!h.pool) h.pool.reset(new Pool);
        ++h.users;
        return true;
    } catch (...) {
        return false;  // copies go through pageable memory
    }
}

void hostcopy_release(int device) {
    std::unique_ptr<Pool> last;  // destroyed after the lock is given up
    std::lock_guard<std::mutex> l(g_pools_m);
    const auto it = pools().find(device);
    if (it == pools().end() || --it->second.users > 0) return;
    last = std::move(it->second.pool);
    pools().erase(it);
}

hipError_t copy_out(int device, hipStream_t stream, const CopyOut* list, int count) {
    try {
        std::vector<CopyOut> items;
        size_t bytes = 0;
        for (int k = 0; k < count; ++k)
            if (list[k].dst && list[k].n) {
                items.push_back(list[k]);
                bytes += 8 * list[k].n;
            }
        if (items.empty()) return hipSuccess;
        if (bytes <= kSlabBytes && items.size() == 1 && items[0].kind == kCopyF64)
            return copy_direct(stream, items[0]);
        Pool* p = pool_of(device);
        Slab slabs[kWorkers];
        if (bytes <= kSlabBytes && items.size() <= kSmallList && p && p->take(slabs, 1) == 1) {
            const hipError_t e = copy_small(slabs[0], stream, items);
            p->give(slabs, 1);
            return e;
        }
        std::vector<Chunk> chunks;
        for (CopyOut& a : items) {
            if (a.kind == kCopyPickF64) {
                int32_t pick = 0;
                hipError_t e = hipMemcpyAsync(&pick, a.pick, sizeof pick, hipMemcpyDeviceToHost, stream);
                const hipError_t done = hipStreamSynchronize(stream);
                if (e == hipSuccess) e = done;
                if (e != hipSuccess) return e;
                if (pick) a.src[0] = a.src[1];
            }
            const size_t per = kChunkBytes / 8;  // 8 B an element at most in a buffer
            for (size_t at = 0; at < a.n; at += per) chunks.push_back({&a, at, a.n - at < per ? a.n - at : per});
        }
        const unsigned hw = std::thread::hardware_concurrency();
        const size_t most = hw > 1 ? std::min<unsigned>(kWorkers, hw / 2) : 1;
        const int want = (int)std::min(most, chunks.size());
        const int few = (int)std::min(most, bytes / (2 * kSlabBytes) + 1);
        // the others' transfers do not wait for the caller's stream by themselves
        if (const hipError_t e = hipStreamSynchronize(stream)) return e;
        hipStream_t streams[2] = {stream, stream};
        const int n = p && bytes > kSlabBytes ? p->take(slabs, want, few, streams) : 0;
        if (n == 0) return copy_plain(stream, chunks, items);
        hipError_t e = hipErrorOutOfMemory;
        try {
            e = copy_long(slabs, n, device, streams, chunks);
        } catch (...) {
        }
        p->give(slabs, n);
        return e;
    } catch (...) {
        return hipErrorOutOfMemory;
    }
}

}  // namespace pic
