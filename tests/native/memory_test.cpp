// The library on a device that has no memory left, and on a host that has
// none (fake_hip.hpp: no GPU is used).
#include "fake_hip.hpp"
#include "qsm_gpu.h"

#include <initializer_list>
#include <new>

namespace {

void fill_up() { dev().capacity = dev().used; }

int failures = 0;
void check(bool ok, const char* what) {
    std::printf("%s: %s\n", what, ok ? "ok" : "FAIL");
    if (!ok) {
        std::printf("  last message: %s\n", qsm_last_error_message());
        ++failures;
    }
}

long alloc_countdown = -1;  // host allocations until one fails; -1: none does

}  // namespace

void* operator new(size_t n) {
    if (alloc_countdown > 0 && --alloc_countdown == 0) throw std::bad_alloc();
    void* p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

double* fake(size_t i) { return reinterpret_cast<double*>(((size_t)1 << 36) + i * kMiB * 64); }
void* const kUserStream = reinterpret_cast<void*>((size_t)77);
const double kZ[3] = {0.0, 0.0, 1.0};

// Two idle blocks of 32 MiB in the pool.
void fill_pool() {
    qsm_release_cached_memory();
    dev().capacity = ~(size_t)0;
    double gbps = 0.0;
    check(qsm_hbm_copy_probe(32 * kMiB, 1, &gbps) == QSM_OK, "probe");
}

void device_memory() {
    void* p = nullptr;
    fill_pool();
    const size_t kept = dev().used;
    check(kept >= 64 * kMiB, "a finished call's blocks are kept");
    fill_up();
    check(qsm_device_alloc(48 * kMiB, &p) == QSM_OK && p, "an allocation that needs the kept blocks");
    check(qsm_device_free(p) == QSM_OK && dev().used == 0, "freed");

    fill_pool();
    fill_up();
    p = fake(1);
    check(qsm_device_alloc(kept + kMiB, &p) == QSM_ENOMEM && !p, "an allocation beyond the device");
    const qsm_grid g = {16, 16, 16, 1.0, 1.0, 1.0};
    check(qsm_dipole_forward(fake(0), &g, kZ, fake(1), kUserStream) == QSM_OK, "the call after it");

    // a stream of the library's own, beside the blocks that the call takes over
    fill_pool();
    check(qsm_dipole_forward(fake(0), &g, kZ, fake(1), kUserStream) == QSM_OK, "on the caller's stream");
    fill_up();
    check(qsm_dipole_forward(fake(0), &g, kZ, fake(1), nullptr) == QSM_OK, "on a stream that needs the kept blocks");

    fill_pool();
    qsm_tv_volume v = {};
    v.grid = g;
    v.bdir[2] = 1.0;
    v.d_field = fake(0);
    v.d_mask = reinterpret_cast<uint8_t*>(fake(1));
    v.d_chi = fake(2);
    const qsm_tv_params prm = {1e-3, 0.1, 0.0, 6};
    qsm_tv_batch* b = nullptr;
    check(qsm_tv_batch_create(&v, 1, &prm, nullptr, &b) == QSM_OK, "batch");
    fill_up();
    check(qsm_tv_batch_run(b, nullptr, nullptr) == QSM_OK && dev().graph_launches == 4,
          "graphs that need the kept blocks");
    qsm_tv_batch_destroy(b);
    dev().capacity = ~(size_t)0;
    qsm_release_cached_memory();
    check(dev().used == 0, "everything given back");
}

// Bytes that a first call with axes of length n sends: the descriptor and the
// FFT tables.  With fail > 0 that call's fail-th host allocation fails first.
size_t table_upload(size_t n, long fail) {
    const qsm_grid g = {n, n, n, 1.0, 1.0, 1.0};
    if (fail > 0) {
        alloc_countdown = fail;
        try {
            (void)qsm_dipole_forward(fake(0), &g, kZ, fake(1), kUserStream);
        } catch (const std::bad_alloc&) {
        }
        alloc_countdown = -1;
    }
    dev().uploaded = 0;
    check(qsm_dipole_forward(fake(0), &g, kZ, fake(1), kUserStream) == QSM_OK, "dipole");
    return dev().uploaded;
}

// Calls whose own host allocations fail, one after the other: handing a block
// back must neither throw nor lose the block, and the entry point without device
// allocations returns a status.
template <class F>
bool stays_in(F&& call) {
    try {
        call();
    } catch (...) {
        alloc_countdown = -1;
        return false;
    }
    alloc_countdown = -1;
    return true;
}
void host_memory() {
    const qsm_grid g = {16, 16, 16, 1.0, 1.0, 1.0};
    qsm_tv_volume v = {};
    v.grid = g;
    v.bdir[2] = 1.0;
    v.d_field = fake(0);
    v.d_mask = reinterpret_cast<uint8_t*>(fake(1));
    v.d_chi = fake(2);
    const qsm_tv_params prm = {1e-3, 0.1, 0.0, 3};
    for (long fail = 1; fail <= 12; ++fail) {
        qsm_release_cached_memory();
        const size_t before = dev().used;
        qsm_tv_batch* b = nullptr;
        check(qsm_tv_batch_create(&v, 1, &prm, nullptr, &b) == QSM_OK, "batch");
        check(stays_in([&] { alloc_countdown = fail; qsm_tv_batch_destroy(b); }), "destroy");
        qsm_release_cached_memory();
        check(dev().used == before, "every block back");
    }
    for (long fail = 1; fail <= 12; ++fail) {
        int rc = -1;
        check(stays_in([&] {
                  alloc_countdown = fail;
                  rc = qsm_dipole_forward_noalloc(fake(0), &g, kZ, fake(1), kUserStream);
              }),
              "without device allocations");
        check(rc == QSM_OK || rc == QSM_ENOMEM, "its status");
        check(qsm_dipole_forward_noalloc(fake(0), &g, kZ, fake(1), kUserStream) == QSM_OK, "and the next call");
    }
}

}  // namespace

int main(int argc, char** argv) {
    if (argc == 2 && !std::strcmp(argv[1], "device")) {
        device_memory();
    } else if (argc == 2 && !std::strcmp(argv[1], "host")) {
        host_memory();
    } else if (argc == 3 && !std::strcmp(argv[1], "tables")) {
        // lengths of every kind of table: register radices, dense, chirp-z
        const long fail = std::atol(argv[2]);
        for (size_t n : {40, 64, 82, 121, 263}) std::printf("upload %zu %zu\n", n, table_upload(n, fail));
    } else {
        return 2;
    }
    std::printf(failures ? "FAILED\n" : "ALL OK\n");
    return failures ? 1 : 0;
}
