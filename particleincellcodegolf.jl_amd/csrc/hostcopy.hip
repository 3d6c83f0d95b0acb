// hostcopy.hip -- device-to-host copies through pinned staging buffers by
// several host threads.
//
// What bounds a copy into ordinary memory is the host: one thread that fills
// pages the caller has never touched and unpacks the mixed formats moves about
// 2 to 7 GB/s, a tenth of the link.  Here each of up to kWorkers threads has two
// pinned buffers; it takes the next chunk of the list, starts
// its transfer into one buffer, and meanwhile unpacks the other into the
// caller's array.  2^24 particles of the mixed 1D run (268 MB) took 64.6 ms
// through one thread and take 6.5 ms.
//
// A list of at most kSmallBytes is one kernel that converts and writes it into
// pinned memory over the link, and one wait: an array at a time, each of its
// transfers and waits costs 20-30 us, and starting the threads 0.2 ms.
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace pic {

namespace {

constexpr int kWorkers = 8;
constexpr int kStreams = 2;
constexpr size_t kChunkBytes = size_t(1) << 20;  // of one pinned buffer
constexpr size_t kSmallBytes = 2 * kChunkBytes;  // the buffers of one worker, which lie together
constexpr int kSmallList = 8;
constexpr int kMaxDevices = 16;

struct Worker {
    hipEvent_t done[2] = {nullptr, nullptr};
    char* pin[2] = {nullptr, nullptr};
};

struct Pool {
    std::mutex m;     // held for the whole of a copy: one at a time per device
    int users = 0;
    int ready = 0;    // workers made so far
    // the workers share two streams: with one, transfers and the waits for
    // them queue behind each other (168 MB in 8.2 ms against 5.2 with eight);
    // each further one costs a process 3 ms when it is first made
    hipStream_t stream[kStreams] = {};
    char* pinned = nullptr;  // the workers' buffers, one allocation
    Worker w[kWorkers];
};
Pool g_pools[kMaxDevices];

void free_pool(Pool& p) {
    for (Worker& w : p.w) {
        for (hipEvent_t& e : w.done)
            if (e) (void)hipEventDestroy(e);
        w = Worker();
    }
    for (hipStream_t& st : p.stream) {
        if (st) (void)hipStreamDestroy(st);
        st = nullptr;
    }
    if (p.pinned) (void)hipHostFree(p.pinned);
    p.pinned = nullptr;
    p.ready = 0;
}

hipError_t make_workers(Pool& p, int n) {
    hipError_t e = hipSuccess;
    for (int k = 0; k < std::min(n, kStreams) && e == hipSuccess; ++k)
        if (!p.stream[k]) e = hipStreamCreateWithFlags(&p.stream[k], hipStreamNonBlocking);
    if (e == hipSuccess && !p.pinned)
        e = hipHostMalloc(reinterpret_cast<void**>(&p.pinned), kWorkers * 2 * kChunkBytes, hipHostMallocDefault);
    for (; e == hipSuccess && p.ready < n; p.ready += e == hipSuccess ? 1 : 0) {
        Worker& w = p.w[p.ready];
        for (int k = 0; k < 2 && e == hipSuccess; ++k) {
            w.pin[k] = p.pinned + (2 * (size_t)p.ready + k) * kChunkBytes;
            if (!w.done[k]) e = hipEventCreateWithFlags(&w.done[k], hipEventDisableTiming);
        }
    }
    return e;
}

size_t element_bytes(CopyKind k) { return k == kCopyF64 || k == kCopyPickF64 ? 8 : 4; }
int sources(CopyKind k) { return k == kCopyPair32 ? 2 : 1; }

struct Chunk {
    const CopyOut* a;
    size_t at, n;
};

void unpack(const Chunk& c, const char* pin) {
    double* o = c.a->dst + c.at;
    const size_t n = c.n;
    switch (c.a->kind) {
    case kCopyF64:
    case kCopyPickF64:
        std::memcpy(o, pin, 8 * n);
        break;
    case kCopyFix32: {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(pin);
        for (size_t j = 0; j < n; ++j) o[j] = (double)q[j] * 0x1p-32;
        break;
    }
    case kCopyUnimod32: {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(pin);
        for (size_t j = 0; j < n; ++j) o[j] = q[j] ? (double)q[j] * 0x1p-32 : 1.0;
        break;
    }
    case kCopyPair32: {
        const float* h = reinterpret_cast<const float*>(pin);
        const float* l = h + n;
        const double s = c.a->scale;
        for (size_t j = 0; j < n; ++j) o[j] = ((double)h[j] + (double)l[j]) * s;
        break;
    }
    }
}

// Chunks off the shared counter until none is left; one transfer ahead.
void work(const Worker& w, hipStream_t stream, int device, const std::vector<Chunk>& chunks, std::atomic<size_t>& next,
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
            size_t off = 0;
            for (int k = 0; k < sources(c->a->kind) && e == hipSuccess; ++k) {
                const size_t b = element_bytes(c->a->kind);
                e = hipMemcpyAsync(w.pin[s] + off, static_cast<const char*>(c->a->src[k]) + b * c->at, b * c->n,
                                   hipMemcpyDeviceToHost, stream);
                off += b * c->n;
            }
            if (e == hipSuccess) e = hipEventRecord(w.done[s], stream);
        }
        if (flying && e == hipSuccess) {
            e = hipEventSynchronize(w.done[s ^ 1]);
            if (e == hipSuccess) unpack(*flying, w.pin[s ^ 1]);
        }
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(stream);  // nothing may write the buffers later
            return fail(e);
        }
        if (!c) return;
        flying = c;
    }
}

// A short list converted straight into pinned memory; off[k]: the first output
// element of array k.
struct SmallList {
    CopyOut a[kSmallList];
    size_t off[kSmallList + 1];
    int n;
};

__global__ void __launch_bounds__(256) k_copy_small(SmallList l, double* __restrict__ out) {
    const size_t total = l.off[l.n];
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        int k = 0;
        while (i >= l.off[k + 1]) ++k;
        const CopyOut& a = l.a[k];
        const size_t j = i - l.off[k];
        double v;
        if (a.kind == kCopyF64) {
            v = static_cast<const double*>(a.src[0])[j];
        } else if (a.kind == kCopyPickF64) {
            v = static_cast<const double*>(a.src[*a.pick ? 1 : 0])[j];
        } else if (a.kind == kCopyPair32) {
            v = ((double)static_cast<const float*>(a.src[0])[j] + (double)static_cast<const float*>(a.src[1])[j]) * a.scale;
        } else {
            const uint32_t q = static_cast<const uint32_t*>(a.src[0])[j];
            v = a.kind == kCopyUnimod32 && q == 0 ? 1.0 : (double)q * 0x1p-32;
        }
        out[i] = v;
    }
}

hipError_t copy_small(const Worker& w, hipStream_t stream, const SmallList& l) {
    const size_t total = l.off[l.n];
    const unsigned blocks = (unsigned)std::min<size_t>((total + 255) / 256, 512);
    k_copy_small<<<blocks, 256, 0, stream>>>(l, reinterpret_cast<double*>(w.pin[0]));
    hipError_t e = hipGetLastError();
    const hipError_t done = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = done;
    if (e != hipSuccess) return e;
    for (int k = 0; k < l.n; ++k) std::memcpy(l.a[k].dst, w.pin[0] + 8 * l.off[k], 8 * l.a[k].n);
    return hipSuccess;
}

}  // namespace

void hostcopy_retain(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    std::lock_guard<std::mutex> l(g_pools[device].m);
    ++g_pools[device].users;
}

void hostcopy_release(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    Pool& p = g_pools[device];
    std::lock_guard<std::mutex> l(p.m);
    if (p.users > 0 && --p.users > 0) return;
    free_pool(p);
}

hipError_t copy_out(int device, const CopyOut* list, int count) {
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    try {
        std::vector<CopyOut> items;
        size_t bytes = 0;
        for (int k = 0; k < count; ++k)
            if (list[k].dst && list[k].n) {
                items.push_back(list[k]);
                bytes += 8 * list[k].n;
            }
        if (items.empty()) return hipSuccess;
        Pool& p = g_pools[device];
        std::lock_guard<std::mutex> lock(p.m);
        if (bytes <= kSmallBytes && items.size() <= kSmallList) {
            if (const hipError_t e = make_workers(p, 1)) return e;
            SmallList l{};
            for (const CopyOut& a : items) {
                l.a[l.n] = a;
                l.off[l.n + 1] = l.off[l.n] + a.n;
                ++l.n;
            }
            return copy_small(p.w[0], p.stream[0], l);
        }
        std::vector<Chunk> chunks;
        for (CopyOut& a : items) {
            if (a.kind == kCopyPickF64) {
                int32_t pick = 0;
                if (const hipError_t e = hipMemcpy(&pick, a.pick, sizeof pick, hipMemcpyDeviceToHost)) return e;
                if (pick) a.src[0] = a.src[1];
            }
            const size_t per = kChunkBytes / 8;  // 8 B an element at most in a buffer
            for (size_t at = 0; at < a.n; at += per) chunks.push_back({&a, at, a.n - at < per ? a.n - at : per});
        }
        const unsigned hw = std::thread::hardware_concurrency();
        int n = (int)std::min<size_t>(chunks.size(), hw > 1 ? std::min<unsigned>(kWorkers, hw / 2) : 1);
        const hipError_t made = make_workers(p, n);
        if (made != hipSuccess && p.ready == 0) return made;
        n = std::min(n, p.ready);
        std::atomic<size_t> next(0);
        std::atomic<int> error(hipSuccess);
        std::vector<std::thread> threads;
        try {
            for (int k = 1; k < n; ++k)
                threads.emplace_back([&, k] { work(p.w[k], p.stream[k % kStreams], device, chunks, next, error); });
        } catch (...) {
            // fewer threads than asked for: the others take their chunks
        }
        work(p.w[0], p.stream[0], device, chunks, next, error);
        for (std::thread& t : threads) t.join();
        return (hipError_t)error.load();
    } catch (...) {
        return hipErrorOutOfMemory;
    }
}

}  // namespace pic
