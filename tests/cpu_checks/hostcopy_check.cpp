// Host check of csrc/hostcopy.cpp with a stand-in for the HIP calls it makes
// ("device" memory is host memory): every format at the sizes where the path
// changes, what is held and given back, a copy beside one that is stuck in its
// transfers, and the copies that find no staging memory.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "hostcopy.h"

using namespace pic;

// ---- the stand-in -----------------------------------------------------------
static std::mutex fake_m;
static std::condition_variable fake_cv;
static std::map<void*, size_t> fake_pins;
static size_t fake_pinned = 0, fake_most = 0;
static int fake_streams = 0, fake_events = 0;
static bool fail_pin = false, fail_stream = false, fail_event = false, fail_copy = false;
static std::atomic<const void*> gate_from{nullptr}, gate_to{nullptr};  // transfers from here wait
static int gate_waiting = 0;

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::mutex> l(fake_m);
    if (fail_pin) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    fake_pins[*p] = n;
    fake_pinned += n;
    fake_most = fake_pinned > fake_most ? fake_pinned : fake_most;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> l(fake_m);
    fake_pinned -= fake_pins.at(p);
    fake_pins.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    if (fail_stream) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> l(fake_m);
    *s = reinterpret_cast<hipStream_t>((size_t)(100 + ++fake_streams));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) {
    std::lock_guard<std::mutex> l(fake_m);
    --fake_streams;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (fail_event) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> l(fake_m);
    *e = reinterpret_cast<hipEvent_t>((size_t)(1000 + ++fake_events));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) {
    std::lock_guard<std::mutex> l(fake_m);
    --fake_events;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (fail_copy) return hipErrorUnknown;
    if (s >= gate_from && s < gate_to) {
        std::unique_lock<std::mutex> l(fake_m);
        ++gate_waiting;
        fake_cv.notify_all();
        fake_cv.wait(l, [&] { return !(s >= gate_from && s < gate_to); });
        --gate_waiting;
    }
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
}

namespace pic {
hipError_t launch_copy_small(const SmallList& l, double* out, hipStream_t) {
    for (int k = 0; k < l.n; ++k) {
        const CopyOut& a = l.a[k];
        for (size_t j = 0; j < a.n; ++j) {
            double v;
            if (a.kind == kCopyF64) v = static_cast<const double*>(a.src[0])[j];
            else if (a.kind == kCopyPickF64) v = static_cast<const double*>(a.src[*a.pick ? 1 : 0])[j];
            else if (a.kind == kCopyPair32)
                v = ((double)static_cast<const float*>(a.src[0])[j] + (double)static_cast<const float*>(a.src[1])[j]) * a.scale;
            else {
                const uint32_t q = static_cast<const uint32_t*>(a.src[0])[j];
                v = a.kind == kCopyUnimod32 && q == 0 ? 1.0 : (double)q * 0x1p-32;
            }
            out[l.off[k] + j] = v;
        }
    }
    return hipSuccess;
}
}  // namespace pic

// ---- the checks -------------------------------------------------------------
static int bad = 0;
static void expect(bool ok, const char* what, long long at = 0) {
    if (!ok && bad++ < 20) std::printf("not so: %s (%lld)\n", what, at);
}

struct Data {
    std::vector<double> f, g;
    std::vector<uint32_t> q;
    std::vector<float> h, l;
    int32_t pick = 1;
    explicit Data(size_t n) : f(n), g(n), q(n), h(n), l(n) {
        for (size_t i = 0; i < n; ++i) {
            f[i] = 0.5 + (double)i;
            g[i] = -1.0 - (double)i;
            q[i] = i % 5 ? (uint32_t)(i * 2654435761u) : 0;
            h[i] = 3.0f + (float)i;
            l[i] = 1e-9f * (float)(i % 91);
        }
    }
};

// every format in one list; its outputs
static void roundtrip(int device, size_t n, const char* what) {
    Data d(n);
    std::vector<double> o(5 * n, -7.0);
    const CopyOut list[6] = {{kCopyF64, o.data(), {d.f.data(), nullptr}, n, 1.0, nullptr},
                             {kCopyFix32, o.data() + n, {d.q.data(), nullptr}, n, 1.0, nullptr},
                             {kCopyF64, nullptr, {d.f.data(), nullptr}, n, 1.0, nullptr},
                             {kCopyUnimod32, o.data() + 2 * n, {d.q.data(), nullptr}, n, 1.0, nullptr},
                             {kCopyPair32, o.data() + 3 * n, {d.h.data(), d.l.data()}, n, 0.125, nullptr},
                             {kCopyPickF64, o.data() + 4 * n, {d.f.data(), d.g.data()}, n, 1.0, &d.pick}};
    expect(copy_out(device, nullptr, list, 6) == hipSuccess, what, (long long)n);
    size_t wrong = 0;
    for (size_t i = 0; i < n; ++i) {
        wrong += o[i] != d.f[i];
        wrong += o[n + i] != (double)d.q[i] * 0x1p-32;
        wrong += o[2 * n + i] != (d.q[i] ? (double)d.q[i] * 0x1p-32 : 1.0);
        wrong += o[3 * n + i] != ((double)d.h[i] + (double)d.l[i]) * 0.125;
        wrong += o[4 * n + i] != d.g[i];
    }
    expect(wrong == 0, what, (long long)n);
}

static const size_t sizes[] = {1, 1000, 52428, 52429, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, 1000003};

static void formats(int device, const char* what) {
    for (size_t n : sizes) roundtrip(device, n, what);
}

// a copy while another's transfers are stuck
static void beside(int device, size_t n) {
    Data a(1 << 20), b(n);
    std::vector<double> oa(a.f.size()), ob(n);
    {
        std::lock_guard<std::mutex> l(fake_m);
        gate_from = a.f.data();
        gate_to = a.f.data() + a.f.size();
    }
    auto copy = [device](const Data& d, std::vector<double>& o) {
        const CopyOut c = {kCopyF64, o.data(), {d.f.data(), nullptr}, o.size(), 1.0, nullptr};
        return copy_out(device, nullptr, &c, 1);
    };
    auto stuck = std::async(std::launch::async, [&] { return copy(a, oa); });
    {
        std::unique_lock<std::mutex> l(fake_m);
        fake_cv.wait(l, [] { return gate_waiting > 0; });
    }
    auto other = std::async(std::launch::async, [&] { return copy(b, ob); });
    const bool through = other.wait_for(std::chrono::seconds(20)) == std::future_status::ready;
    expect(through, "a copy beside a stuck one ends", (long long)n);
    expect(stuck.wait_for(std::chrono::seconds(0)) != std::future_status::ready, "the stuck copy is stuck");
    {
        std::lock_guard<std::mutex> l(fake_m);
        gate_from = nullptr;
        gate_to = nullptr;
    }
    fake_cv.notify_all();
    expect(stuck.get() == hipSuccess && other.get() == hipSuccess, "both copies end");
    expect(oa == a.f && ob == b.f, "both copies hold their data", (long long)n);
}

int main() {
    // formats and sizes, and what a short list pins
    expect(hostcopy_retain(0), "retained");
    roundtrip(0, 1000, "a short list");
    expect(fake_most <= (2u << 20), "a short list pins one slab", (long long)fake_most);
    formats(0, "formats");
    for (size_t n : {(size_t)1000, (size_t)1 << 19}) beside(0, n);
    std::vector<std::thread> ts;
    for (int k = 0; k < 6; ++k) ts.emplace_back([] { formats(0, "six threads"); });
    for (std::thread& t : ts) t.join();
    expect(fake_most <= (32u << 20), "at most 32 MiB are pinned", (long long)fake_most);
    // given back with the last user, and made again
    expect(hostcopy_retain(0), "retained again");
    hostcopy_release(0);
    expect(fake_pinned > 0, "kept for the other user");
    hostcopy_release(0);
    expect(fake_pinned == 0 && fake_streams == 0 && fake_events == 0, "all given back");
    expect(hostcopy_retain(0), "retained after that");
    formats(0, "made again");
    // an error in a transfer is reported, and the slabs come back
    for (int k = 0; k < 40; ++k) {
        Data d(1 << 19);
        std::vector<double> o(d.f.size());
        const CopyOut c = {kCopyF64, o.data(), {d.f.data(), nullptr}, o.size(), 1.0, nullptr};
        fail_copy = true;
        expect(copy_out(0, nullptr, &c, 1) == hipErrorUnknown, "the transfer's error");
        fail_copy = false;
    }
    formats(0, "after errors");
    hostcopy_release(0);
    expect(fake_pinned == 0 && fake_streams == 0 && fake_events == 0, "all given back after errors");
    // without pinned memory, events or the second stream
    for (bool* f : {&fail_pin, &fail_event, &fail_stream}) {
        *f = true;
        expect(hostcopy_retain(0), "retained");
        formats(0, f == &fail_pin ? "no pinned memory" : f == &fail_event ? "no events" : "no second stream");
        *f = false;
        hostcopy_release(0);
    }
    expect(fake_pinned == 0 && fake_streams == 0 && fake_events == 0, "nothing is left");
    // no context holds the buffers
    formats(0, "not retained");
    // every ordinal that a context may name
    for (int device : {15, 16, 63}) {
        expect(hostcopy_retain(device), "retained", device);
        formats(device, "device");
        expect(fake_pinned > 0, "staged", device);
        hostcopy_release(device);
    }
    expect(fake_pinned == 0 && fake_streams == 0 && fake_events == 0, "nothing is left");
    std::printf("%d wrong\n", bad);
    return bad != 0;
}
