// HIP for test programs of the library that use no GPU: defined in the program,
// these functions take the place of the runtime's.  Device memory is counted
// against a capacity that the test sets, uploads are counted, launches recorded
// by name and number of blocks; kernels do nothing.
#pragma once

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

struct Dim3 {
    unsigned x, y, z;
};

namespace {

enum { kSuccess = 0, kOutOfMemory = 2 };
constexpr size_t kMiB = (size_t)1 << 20, kStreamCost = kMiB, kGraphCost = kMiB;
// (function-local, never destroyed: the library may free after main)
struct Device {
    size_t capacity = ~(size_t)0, used = 0, uploaded = 0;
    std::map<void*, size_t> blocks;
    int last_error = kSuccess, graph_launches = 0;
    std::map<const void*, std::string> kernels;            // by host function
    std::vector<std::pair<std::string, unsigned>> launches;  // kernel, blocks
    Dim3 grid = {}, block = {};
    long next_id = 1;
};
Device& dev() {
    static Device* d = new Device();
    return *d;
}
bool charge(size_t bytes) {
    Device& d = dev();
    if (d.capacity - d.used < bytes) {
        d.last_error = kOutOfMemory;
        return false;
    }
    d.used += bytes;
    return true;
}

}  // namespace

extern "C" {
int hipGetDevice(int* d) { *d = 0; return kSuccess; }
int hipGetLastError() {
    const int e = dev().last_error;
    dev().last_error = kSuccess;
    return e;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : e ? "error" : "no error"; }
int hipMalloc(void** p, size_t n) {
    if (!charge(n)) return kOutOfMemory;
    *p = reinterpret_cast<void*>(((size_t)1 << 40) + kMiB * 1024 * (size_t)dev().next_id++);
    dev().blocks[*p] = n;
    return kSuccess;
}
int hipFree(void* p) {
    auto it = dev().blocks.find(p);
    if (it == dev().blocks.end()) return 1;
    dev().used -= it->second;
    dev().blocks.erase(it);
    return kSuccess;
}
int hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(n, 1); return *p ? kSuccess : kOutOfMemory; }
int hipHostFree(void* p) { std::free(p); return kSuccess; }
int hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return kSuccess; }
int hipStreamCreateWithFlags(void** s, unsigned) {
    if (!charge(kStreamCost)) return kOutOfMemory;
    *s = reinterpret_cast<void*>(dev().next_id++);
    return kSuccess;
}
int hipStreamDestroy(void*) { dev().used -= kStreamCost; return kSuccess; }
int hipStreamSynchronize(void*) { return kSuccess; }
int hipStreamWaitEvent(void*, void*, unsigned) { return kSuccess; }
int hipStreamIsCapturing(void*, int* s) { *s = 0; return kSuccess; }
int hipStreamBeginCapture(void*, int) { return kSuccess; }
int hipStreamEndCapture(void*, void** g) { *g = reinterpret_cast<void*>(dev().next_id++); return kSuccess; }
int hipGraphInstantiate(void** x, void*, void**, char*, size_t) {
    if (!charge(kGraphCost)) return kOutOfMemory;
    *x = reinterpret_cast<void*>(dev().next_id++);
    return kSuccess;
}
int hipGraphDestroy(void*) { return kSuccess; }
int hipGraphExecDestroy(void*) { dev().used -= kGraphCost; return kSuccess; }
int hipGraphLaunch(void*, void*) { ++dev().graph_launches; return kSuccess; }
int hipEventCreate(void** e) { *e = reinterpret_cast<void*>(dev().next_id++); return kSuccess; }
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) { return kSuccess; }
int hipEventRecord(void*, void*) { return kSuccess; }
int hipEventSynchronize(void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 1.0f; return kSuccess; }
int hipGetSymbolAddress(void** p, const void*) { *p = reinterpret_cast<void*>((size_t)1 << 38); return kSuccess; }
int hipDeviceSynchronize() { return kSuccess; }
int hipMemcpy(void*, const void*, size_t n, int) { dev().uploaded += n; return kSuccess; }
int hipMemcpyAsync(void*, const void*, size_t n, int, void*) { dev().uploaded += n; return kSuccess; }
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    dev().kernels[f] = name;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void**, size_t, void*) {
    dev().launches.emplace_back(dev().kernels[f], grid.x);
    return kSuccess;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t, void*) {
    dev().grid = grid;
    dev().block = block;
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* n, void** s) {
    *grid = dev().grid;
    *block = dev().block;
    *n = 0;
    *s = nullptr;
    return kSuccess;
}
}
