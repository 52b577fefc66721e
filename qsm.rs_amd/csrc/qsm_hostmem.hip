// Device workspaces, streams, pinned blocks and host copies (qsm_hostmem.hpp).
//
// Why: the host-pointer entry points spend their time outside the kernels.
// Measured for a 192x192x128 volume (38 MB in f64): a pageable hipMemcpy to
// the device 1.3 ms, from the device 2.1-4.4 ms (half of it the host's page
// faults in a fresh array), against 1.1 and 0.8 ms narrowed through pinned
// chunks; hipMalloc and hipFree of its buffers, with a device-wide wait, and
// the FFT tables 0.2-0.5 ms; the kernels of a closed-form inversion 0.1 ms.
#include "qsm_hostmem.hpp"

#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <cerrno>
#include <cstdint>
#include <cstring>
#include <list>
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

namespace qsm {
namespace {

struct Block {
    void* p;
    size_t bytes;
    int dev;
};

constexpr size_t kStreamsKept = 8, kPinnedKept = 64;
constexpr size_t kChunk = (size_t)2 << 20;  // bytes of one staging buffer
constexpr int kLanesKept = 4;  // per device: calls of as many threads copy at once

// A pair of staging buffers.  A copy's chunks alternate between them; ev[i]
// marks the last device copy of buf[i].
struct Lane {
    char* buf[2] = {};
    hipEvent_t ev[2] = {};
    hipStream_t stream = nullptr;
    int dev = -1;
};

struct Store {
    std::mutex mu;
    std::unordered_map<void*, Block> live;  // blocks handed out
    std::list<Block> kept;                  // idle blocks, oldest first
    size_t kept_bytes = 0;
    std::unordered_map<hipStream_t, int> stream_dev;          // streams made here
    std::vector<std::pair<int, hipStream_t>> streams;         // idle ones
    std::vector<void*> pinned;
    std::vector<Lane> lanes;                                  // idle lanes
};

// Adds to one of the store's containers; false where the host has no memory for
// that, and the caller gives the object back to the runtime instead.  (Nothing
// here throws: these are the calls that free.)
template <class F>
bool kept_by(F&& add) noexcept {
    try {
        add();
        return true;
    } catch (const std::bad_alloc&) {
        return false;
    }
}

// Never destroyed: the runtime may be gone when static objects are.
Store& store() {
    static Store* s = new Store();
    return *s;
}

// Sizes are rounded so that volumes of about the same size share blocks.
size_t rounded(size_t bytes) {
    const size_t g = bytes < ((size_t)1 << 20) ? (size_t)4096 : (size_t)1 << 20;
    return (std::max<size_t>(bytes, 1) + g - 1) / g * g;
}

void lane_destroy(Lane& l) {
    for (int i = 0; i < 2; ++i) {
        if (l.ev[i]) (void)hipEventDestroy(l.ev[i]);
        if (l.buf[i]) (void)hipHostFree(l.buf[i]);
    }
    if (l.stream) (void)hipStreamDestroy(l.stream);
    l = Lane{};
}

hipError_t lane_take(int dev, Lane& out) {
    {
        Store& s = store();
        std::lock_guard<std::mutex> lk(s.mu);
        for (size_t i = 0; i < s.lanes.size(); ++i)
            if (s.lanes[i].dev == dev) {
                out = s.lanes[i];
                s.lanes.erase(s.lanes.begin() + i);
                return hipSuccess;
            }
    }
    Lane l;
    l.dev = dev;
    hipError_t e = with_trim([&] { return hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking); });
    if (e != hipSuccess) l.stream = nullptr;
    for (int i = 0; i < 2 && e == hipSuccess; ++i) {
        e = with_trim([&] { return hipHostMalloc((void**)&l.buf[i], kChunk, hipHostMallocDefault); });
        if (e != hipSuccess) l.buf[i] = nullptr;
        if (e == hipSuccess) {
            e = hipEventCreateWithFlags(&l.ev[i], hipEventDisableTiming);
            if (e != hipSuccess) l.ev[i] = nullptr;
        }
    }
    if (e != hipSuccess) {
        lane_destroy(l);
        return e;
    }
    out = l;
    return hipSuccess;
}

// An idle lane back.
void lane_give(Lane& l) {
    Store& s = store();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        int have = 0;
        for (const Lane& k : s.lanes) have += k.dev == l.dev;
        if (have < kLanesKept && kept_by([&] { s.lanes.push_back(l); })) return;
    }
    lane_destroy(l);
}

// Host side of a chunk: bytes as they are, or f64 on the host and f32 on the
// device (the kernels' own first and last conversion, made here so that half
// the bytes cross the link).
void fill_chunk(char* buf, const char* src, size_t bytes, bool narrow) {
    if (!narrow) {
        std::memcpy(buf, src, bytes);
        return;
    }
    float* d = reinterpret_cast<float*>(buf);
    const double* f = reinterpret_cast<const double*>(src);
    for (size_t i = 0; i < bytes / sizeof(float); ++i) d[i] = (float)f[i];
}
void drain_chunk(char* dst, const char* buf, size_t bytes, bool narrow) {
    if (!narrow) {
        std::memcpy(dst, buf, bytes);
        return;
    }
    // Stores past the caches: an ordinary store reads its line of the result
    // array, which is larger than the caches, from memory first (38 MB of
    // doubles: 4.0 ms, so 0.8).
    typedef double d2 __attribute__((ext_vector_type(2)));
    double* d = reinterpret_cast<double*>(dst);
    const float* f = reinterpret_cast<const float*>(buf);
    const size_t n = bytes / sizeof(float);
    size_t i = 0;
    for (; i < n && (uintptr_t)(d + i) % sizeof(d2); ++i) d[i] = (double)f[i];
    for (; i + 2 <= n; i += 2) {
        const d2 v = {(double)f[i], (double)f[i + 1]};
        __builtin_nontemporal_store(v, reinterpret_cast<d2*>(d + i));
    }
    for (; i < n; ++i) d[i] = (double)f[i];
    __builtin_ia32_sfence();
}

// bytes: on the device.  One thread: with two to six a 38 MB upload takes
// 0.5-0.7 ms instead of 1.1 where the CPUs are idle, but where the caller's
// program keeps a spinning thread pool (an OpenMP runtime between two
// parallel regions) the helpers wait for a CPU with a chunk in hand, and the
// same round trip took 4.5-7.2 ms instead of 4.3.
hipError_t copy_staged(bool to_device, void* dst_, const void* src_, size_t bytes, bool narrow) {
    if (!bytes) return hipSuccess;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    Lane l;
    if ((e = lane_take(dev, l)) != hipSuccess) return e;
    char* dst = static_cast<char*>(dst_);
    const char* src = static_cast<const char*>(src_);
    const size_t nchunk = (bytes + kChunk - 1) / kChunk, host_chunk = kChunk * (narrow ? 2 : 1);
    auto len = [&](size_t k) { return std::min(kChunk, bytes - k * kChunk); };
    size_t pend[2] = {};  // chunk in flight to the host, per buffer
    bool busy[2] = {};
    auto drain = [&](int i) {  // waits for buf[i]'s device copy; to the host: hands its chunk over
        if (!busy[i]) return hipSuccess;
        const hipError_t w = hipEventSynchronize(l.ev[i]);
        if (w == hipSuccess && !to_device) drain_chunk(dst + pend[i] * host_chunk, l.buf[i], len(pend[i]), narrow);
        busy[i] = false;
        return w;
    };
    int i = 0;
    for (size_t k = 0; k < nchunk && e == hipSuccess; ++k, i ^= 1) {
        if ((e = drain(i)) != hipSuccess) break;
        if (to_device) {
            fill_chunk(l.buf[i], src + k * host_chunk, len(k), narrow);
            e = hipMemcpyAsync(dst + k * kChunk, l.buf[i], len(k), hipMemcpyHostToDevice, l.stream);
        } else {
            e = hipMemcpyAsync(l.buf[i], src + k * kChunk, len(k), hipMemcpyDeviceToHost, l.stream);
        }
        if (e != hipSuccess) break;
        if ((e = hipEventRecord(l.ev[i], l.stream)) != hipSuccess) break;
        pend[i] = k;
        busy[i] = true;
    }
    for (int q = 0; q < 2; ++q, i ^= 1) {  // the older one first
        const hipError_t w = drain(i);
        if (e == hipSuccess) e = w;
    }
    if (e == hipSuccess) {
        lane_give(l);
    } else {
        (void)hipStreamSynchronize(l.stream);
        lane_destroy(l);
    }
    return e;
}

}  // namespace

hipError_t workspace_alloc(void** p, size_t bytes) {
    *p = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const size_t want = rounded(bytes);
    Store& s = store();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        auto best = s.kept.end();
        for (auto it = s.kept.begin(); it != s.kept.end(); ++it)
            if (it->dev == dev && it->bytes >= want && it->bytes <= want + want / 4 &&
                (best == s.kept.end() || it->bytes < best->bytes))
                best = it;
        if (best != s.kept.end()) {
            if (!kept_by([&] { s.live.emplace(best->p, *best); })) return hipErrorOutOfMemory;
            *p = best->p;
            s.kept_bytes -= best->bytes;
            s.kept.erase(best);
            return hipSuccess;
        }
    }
    e = with_trim([&] { return hipMalloc(p, want); });
    if (e != hipSuccess) {
        *p = nullptr;
        return e;
    }
    bool known;
    {
        std::lock_guard<std::mutex> lk(s.mu);
        known = kept_by([&] { s.live.emplace(*p, Block{*p, want, dev}); });
    }
    if (known) return hipSuccess;
    (void)hipFree(*p);
    *p = nullptr;
    return hipErrorOutOfMemory;
}

void workspace_free(void* p) {
    if (!p) return;
    Store& s = store();
    std::list<Block> back, node;
    const bool noted = kept_by([&] { node.emplace_back(); });
    {
        std::lock_guard<std::mutex> lk(s.mu);
        auto it = s.live.find(p);
        if (it == s.live.end()) return;  // not one of ours
        const Block b = it->second;
        s.live.erase(it);
        if (noted && b.bytes <= kWorkspaceKept / 2) {
            node.front() = b;
            s.kept.splice(s.kept.end(), node);
            s.kept_bytes += b.bytes;
            while (s.kept_bytes > kWorkspaceKept) {
                s.kept_bytes -= s.kept.front().bytes;
                back.splice(back.end(), s.kept, s.kept.begin());
            }
            p = nullptr;
        }
    }
    if (p) (void)hipFree(p);
    for (const Block& q : back) (void)hipFree(q.p);
}

void workspace_trim() {
    Store& s = store();
    std::list<Block> kept;
    std::vector<std::pair<int, hipStream_t>> streams;
    std::vector<void*> pinned;
    std::vector<Lane> lanes;
    {
        std::lock_guard<std::mutex> lk(s.mu);
        kept.swap(s.kept);
        s.kept_bytes = 0;
        streams.swap(s.streams);
        pinned.swap(s.pinned);
        lanes.swap(s.lanes);
        for (auto& st : streams) s.stream_dev.erase(st.second);
    }
    for (const Block& b : kept) (void)hipFree(b.p);
    for (auto& st : streams) (void)hipStreamDestroy(st.second);
    for (void* q : pinned) (void)hipHostFree(q);
    for (Lane& l : lanes) lane_destroy(l);
}

hipError_t stream_take(hipStream_t* out) {
    *out = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    Store& s = store();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        for (size_t i = 0; i < s.streams.size(); ++i)
            if (s.streams[i].first == dev) {
                *out = s.streams[i].second;
                s.streams.erase(s.streams.begin() + i);
                return hipSuccess;
            }
    }
    e = with_trim([&] { return hipStreamCreateWithFlags(out, hipStreamNonBlocking); });
    if (e != hipSuccess) {
        *out = nullptr;
        return e;
    }
    bool known;
    {
        std::lock_guard<std::mutex> lk(s.mu);
        known = kept_by([&] { s.stream_dev.emplace(*out, dev); });
    }
    if (known) return hipSuccess;
    (void)hipStreamDestroy(*out);
    *out = nullptr;
    return hipErrorOutOfMemory;
}

void stream_give(hipStream_t st) {
    if (!st) return;
    Store& s = store();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        auto it = s.stream_dev.find(st);
        if (it != s.stream_dev.end() && s.streams.size() < kStreamsKept &&
            kept_by([&] { s.streams.emplace_back(it->second, st); }))
            return;
        s.stream_dev.erase(st);
    }
    (void)hipStreamDestroy(st);
}

hipError_t pinned_take(void** p) {
    Store& s = store();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        if (!s.pinned.empty()) {
            *p = s.pinned.back();
            s.pinned.pop_back();
            return hipSuccess;
        }
    }
    const hipError_t e = with_trim([&] {
        return hipHostMalloc(p, kPinnedBlock, hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable);
    });
    if (e != hipSuccess) *p = nullptr;
    return e;
}

void pinned_give(void* p) {
    if (!p) return;
    {
        Store& s = store();
        std::lock_guard<std::mutex> lk(s.mu);
        if (s.pinned.size() < kPinnedKept && kept_by([&] { s.pinned.push_back(p); })) return;
    }
    (void)hipHostFree(p);
}

void prefault(void* p, size_t bytes) {
#ifdef MADV_POPULATE_WRITE
    constexpr int populate = MADV_POPULATE_WRITE;
#else
    constexpr int populate = 23;  // Linux 5.14; an older kernel refuses it
#endif
    const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
    const uintptr_t a = ((uintptr_t)p + page - 1) / page * page, b = ((uintptr_t)p + bytes) / page * page;
    if (bytes < kChunk || b <= a) return;
    const int keep = errno;
    (void)madvise((void*)a, b - a, populate);  // a hint: the copy faults in what this leaves
    errno = keep;
}

hipError_t copy_to_device(void* dst, const void* src, size_t bytes) { return copy_staged(true, dst, src, bytes, false); }
hipError_t copy_to_host(void* dst, const void* src, size_t bytes) { return copy_staged(false, dst, src, bytes, false); }
hipError_t copy_to_device_f32(float* dst, const double* src, size_t n) {
    return copy_staged(true, dst, src, n * sizeof(float), true);
}
hipError_t copy_to_host_f32(double* dst, const float* src, size_t n) {
    return copy_staged(false, dst, src, n * sizeof(float), true);
}

}  // namespace qsm
