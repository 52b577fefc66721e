// The shares of a block in the stages of fft_dense.hpp, for every length that
// runs them and every tile that is launched: a register stage needs a thread's
// place for every butterfly, a dense stage a wave's for every unit, and the tile
// must hold the sequences (work past either end would be dropped).  The tiles of
// 8 elements per thread are also transformed, against a direct DFT in double.
#include "../../qsm.rs_amd/csrc/fft_dense.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace qsmfft;

template <int E>
static int places(int R) {
    switch (R) {
#define PLACES(r) case r: return RegStage<r, E>::B * kThreads;
        PLACES(2) PLACES(3) PLACES(4) PLACES(5) PLACES(6) PLACES(7) PLACES(8) PLACES(9) PLACES(10) PLACES(11)
        PLACES(12) PLACES(13) PLACES(14) PLACES(15) PLACES(16)
        default: return 0;
    }
}

// ncols sequences of length n (columns: interleaved) in tiles of E elements per thread.
template <int E, bool COLFAST>
static bool fits(int n, int ncols) {
    Plan P{};
    if (!make_dense_plan(n, P) || n * ncols > E * kThreads) return false;
    const int es = COLFAST ? ncols : 1, cs = COLFAST ? 1 : n;
    for (int s = 0; s < P.nstages; ++s) {
        if (P.radix[s] <= kMaxRegRadix) {
            const StageGeom g = plan_geom(P, s, ncols, es, cs);
            if (g.nb * g.ncols > places<E>(P.radix[s])) return false;
        } else {
            const DenseGeom g = dense_geom(P, s, ncols, es, cs);
            if (g.units > kDenseUnits * E * kThreads / kDenseElems * (kThreads / 64)) return false;
        }
    }
    return true;
}

// Register stages alone, as the device runs them in tiles of 8 elements.
template <int R, bool COLFAST, int LOG2C>
static void stage8(std::vector<float2>& v, const Plan& P, int s, int ncols, int es, int cs, const float2* tw) {
    const StageGeom g = plan_geom(P, s, ncols, es, cs);
    std::vector<float2> out(v.size(), make_float2(NAN, NAN));
    for (int tid = 0; tid < kThreads; ++tid) {
        float2 r[RegStage<R, 8>::B][R];
        reg_stage_load<R, COLFAST, LOG2C, 8>(v.data(), tid, g, r);
        reg_stage_store<R, COLFAST, LOG2C, false, 8>(out.data(), tid, g, r, tw);
    }
    v = out;
}
template <bool COLFAST, int LOG2C>
static double error8(int n, int ncols) {
    Plan P{};
    make_dense_plan(n, P);
    const int es = COLFAST ? ncols : 1, cs = COLFAST ? 1 : n;
    std::vector<float2> tw(n), v((size_t)n * ncols);
    for (int q = 0; q < n; ++q)
        tw[q] = make_float2((float)std::cos(-2.0 * M_PI * q / n), (float)std::sin(-2.0 * M_PI * q / n));
    srand(n + ncols);
    for (auto& x : v) x = make_float2(rand() / (float)RAND_MAX - 0.5f, rand() / (float)RAND_MAX - 0.5f);
    const std::vector<float2> in = v;
    for (int s = 0; s < P.nstages; ++s) switch (P.radix[s]) {
#define STAGE(r) case r: stage8<r, COLFAST, LOG2C>(v, P, s, ncols, es, cs, tw.data()); break;
            STAGE(2) STAGE(3) STAGE(4) STAGE(5) STAGE(6) STAGE(7) STAGE(8) STAGE(9) STAGE(10) STAGE(11) STAGE(12)
            STAGE(13) STAGE(14) STAGE(15) STAGE(16)
            default: return 0.0;  // (dense stages: bounds above, values in dense_emulation.cpp)
        }
    double err = 0.0, most = 0.0;
    for (int c = 0; c < ncols; c += 3)
        for (int k = 0; k < n; ++k) {
            std::complex<double> a = 0.0;
            for (int e = 0; e < n; ++e) {
                const float2 x = in[e * es + c * cs];
                a += std::complex<double>(x.x, x.y) * std::polar(1.0, -2.0 * M_PI * (double)((long)k * e % n) / n);
            }
            const float2 y = v[k * es + c * cs];
            const double d = std::abs(a - std::complex<double>(y.x, y.y));
            err = d == d ? std::max(err, d) : 1e30;
            most = std::max(most, std::abs(a));
        }
    return err / most;
}

int main() {
    int bad = 0, lengths = 0;
    auto check = [&](bool ok, const char* what, int n, int seqs) {
        if (ok) return;
        std::printf("%s: length %d, %d sequences\n", what, n, seqs);
        ++bad;
    };
    for (int n = 2; n <= kMaxDenseLen; ++n) {
        Plan P{};
        if (!make_dense_plan(n, P)) continue;
        ++lengths;
        int least = n;  // butterflies of its dense stages in one sequence
        for (int s = 0; s < P.nstages; ++s)
            if (P.radix[s] > kMaxRegRadix) least = std::min(least, n / P.radix[s]);
        // rows: any count up to what the tile holds, at most 32
        for (int r = 1; r <= std::min(32, 4096 / n); ++r) check(fits<16, false>(n, r), "rows", n, r);
        for (int r = 1; r <= std::min(32, 2048 / n); ++r) check(fits<8, false>(n, r), "C2R rows", n, r);
        // columns: tiles of 16 up to length 256, of 8 above; half tiles of 8 from
        // 128 to 256 with four butterflies a column or more
        check(n <= 256 ? fits<16, true>(n, 16) : fits<16, true>(n, 8), "columns", n, n <= 256 ? 16 : 8);
        if (n >= 128 && n <= 256 && least >= 4) check(fits<8, true>(n, 8), "half tiles", n, 8);
        if (least == n && n % 7 < 2) {
            check(error8<false, 0>(n, std::min(32, 2048 / n)) < 2e-6, "transform of rows", n, 2048 / n);
            if (n <= 256) check(error8<true, 3>(n, 8) < 2e-6, "transform of columns", n, 8);
        }
    }
    std::printf("%d lengths\n%s\n", lengths, bad ? "FAILED" : "ALL OK");
    return bad ? 1 : 0;
}
