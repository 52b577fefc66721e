// Blocks of the x passes of run-time row lengths (fake_hip.hpp: no GPU is
// used).  A launch whose rows fit one round of 768 resident blocks, three a CU,
// has at most an eighth more (whole matrix tiles); R2C passes of TV have at least
// 96.  (A quarter of the rows a block, the rule for compiled lengths, ran up to
// 1728 blocks of 80 elements: a TV iteration up to a fifth slower; full blocks of
// long rows left half the CUs idle.)
#include "fake_hip.hpp"
#include "qsm_gpu.h"

#include <algorithm>

namespace {

double* fake(size_t i) { return reinterpret_cast<double*>(((size_t)1 << 36) + (i << 32)); }
int failures = 0;

void check(const char* what, const std::string& kernel, size_t n, size_t rows, unsigned blocks, size_t tile,
           unsigned least = 0) {
    const size_t most = std::max<size_t>(1, std::min<size_t>(32, tile / n));
    if (blocks >= least && (rows > 768 * (most & ~(size_t)1) || blocks <= 768 + 96)) return;
    std::printf("%s: %s, %zu columns, %zu rows: %u blocks\n", what, kernel.c_str(), n, rows, blocks);
    ++failures;
}

void volume(size_t nx, size_t ny, size_t nz) {
    const qsm_grid g = {nx, ny, nz, 1.0, 1.0, 1.0};
    const double z[3] = {0.0, 0.0, 1.0};
    const size_t pairs = (ny * nz + 1) / 2;
    auto passes = [&](const char* what, int rc) {
        if (rc != QSM_OK) {
            std::printf("%s: %s\n", what, qsm_last_error_message());
            ++failures;
        }
        int seen = 0;
        for (const auto& l : dev().launches) {
            // (the tiles of the R2C passes, and of the V-SHARP ones, hold 4096 elements)
            if (l.first.find("k_r2c_x") != std::string::npos) check(what, l.first, nx, pairs, l.second, 4096, what[0] == 'T' ? 96 : 48), ++seen;
            if (l.first.find("k_c2r_tv") != std::string::npos) check(what, l.first, nx, pairs, l.second, 2048), ++seen;
            if (l.first.find("k_c2r_vs_select") != std::string::npos)
                check(what, l.first, nx, 2 * pairs, l.second, 4096), ++seen;
        }
        if (seen < 2) ++failures;
        dev().launches.clear();
    };
    qsm_tv_volume v = {};
    v.grid = g;
    v.bdir[2] = 1.0;
    v.d_field = fake(0);
    v.d_mask = reinterpret_cast<uint8_t*>(fake(1));
    v.d_chi = fake(2);
    const qsm_tv_params prm = {1e-3, 0.1, 0.0, 2};
    qsm_tv_batch* b = nullptr;
    int rc = qsm_tv_batch_create(&v, 1, &prm, nullptr, &b);
    if (rc == QSM_OK) rc = qsm_tv_batch_set_graphs(b, 0);
    if (rc == QSM_OK) rc = qsm_tv_batch_run(b, nullptr, nullptr);
    qsm_tv_batch_destroy(b);
    passes("TV", rc);
    const qsm_vsharp_volume vv = {g, fake(0), reinterpret_cast<uint8_t*>(fake(1)), fake(2),
                                  reinterpret_cast<uint8_t*>(fake(3))};
    const double radii[2] = {3.0, 2.0};
    qsm_vsharp_batch* s = nullptr;
    rc = qsm_vsharp_batch_create(&vv, 1, radii, 2, 0.05, nullptr, &s);
    if (rc == QSM_OK) rc = qsm_vsharp_batch_run(s, nullptr, nullptr);
    qsm_vsharp_batch_destroy(s);
    passes("V-SHARP", rc);
    passes("dipole", qsm_dipole_forward(fake(0), &g, z, fake(2), nullptr));
}

}  // namespace

int main() {
    // register radices only; one, two, four and eight rows of matrix tiles;
    // one to seventeen butterflies a row; tiles of 8 to 32 rows
    for (size_t n : {20, 33, 65, 82, 104, 125, 143, 164, 205, 211, 231, 251, 289, 338, 398, 429, 507}) {
        volume(n, 64, 48);
        volume(n, 144, 96);
        volume(n, 240, 168);
    }
    std::printf(failures ? "FAILED\n" : "ALL OK\n");
    return failures ? 1 : 0;
}
