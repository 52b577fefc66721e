// CPU emulation of the run-time-length transforms of fft_dense.hpp: every
// thread of the register-radix stages and every lane of the dense stages, with
// the device's index functions, against a direct DFT in double.  Every LDS
// index is checked and every output must be written exactly once.
#include "../../qsm.rs_amd/csrc/fft_dense.hpp"

#include <algorithm>
#include <array>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace qsmfft;

struct Tile {
    std::vector<float2> v;
    std::vector<int> writes;
    bool ok = true;
    float2 get(int i) {
        if (i < 0 || i >= (int)v.size()) { ok = false; return make_float2(NAN, NAN); }
        return v[i];
    }
    void put(std::vector<float2>& out, int i, float2 x) {
        if (i < 0 || i >= (int)v.size()) { ok = false; return; }
        out[i] = x;
        ++writes[i];
    }
};

template <int R, bool COLFAST, int LOG2C, bool INV>
static void emu_reg(Tile& T, const Plan& P, int s, int ncols, int es, int cs, const float2* tw) {
    const StageGeom g = plan_geom(P, s, ncols, es, cs);
    if (g.nb * g.ncols > RegStage<R>::B * kThreads) T.ok = false;  // every butterfly has a thread
    std::vector<float2> out(T.v.size(), make_float2(NAN, NAN));
    for (int tid = 0; tid < kThreads; ++tid) {
        float2 v[RegStage<R>::B][R];
        reg_stage_load<R, COLFAST, LOG2C>(T.v.data(), tid, g, v);
        reg_stage_store<R, COLFAST, LOG2C, INV>(out.data(), tid, g, v, tw);
    }
    T.v = out;
}

template <bool COLFAST, int LOG2C, bool INV>
static void emu_dense(Tile& T, const Plan& P, int s, int ncols, int es, int cs, const float2* tw) {
    const DenseGeom g = dense_geom(P, s, ncols, es, cs);
    if (g.units > kDenseUnits * (kThreads / 64)) T.ok = false;
    std::vector<float2> coef(dense_table_len(g.R)), out(T.v.size(), make_float2(NAN, NAN));
    dense_table(g.R, coef.data());
    T.writes.assign(T.v.size(), 0);
    for (int unit = 0; unit < g.units; ++unit) {
        int nt, mt;
        dense_unit(g, unit, nt, mt);
        if (nt != unit / g.mt || mt != unit % g.mt) T.ok = false;
        // operands of each lane, then the 16 x 16 results (row: coefficient
        // lane & 15, column: item lane & 15, r by lane >> 4)
        std::vector<std::array<float, 4>> acc(256, std::array<float, 4>{0.0f, 0.0f, 0.0f, 0.0f}), sum(256);
        for (int lane = 0; lane < 64; ++lane) {
            int in, o, ts;
            dense_item<COLFAST, LOG2C>(g, std::min(nt * 16 + (lane & 15), g.items - 1), in, o, ts);
            const float2 x0 = T.get(in);
            if (lane < 16)
                for (int row = 0; row < 16; ++row) sum[row * 16 + lane] = {x0.x, x0.y, 0.0f, 0.0f};
        }
        auto close_block = [&] {
            for (int i = 0; i < 256; ++i)
                for (int q = 0; q < 4; ++q) {
                    sum[i][q] += acc[i][q];
                    acc[i][q] = 0.0f;
                }
        };
        for (int kk = 0; kk < g.kb * kDenseBlock; ++kk) {
            if (kk != 0 && kk % kDenseBlock == 0) close_block();
            for (int lane = 0; lane < 64; ++lane) {
                int in, o, ts;
                dense_item<COLFAST, LOG2C>(g, std::min(nt * 16 + (lane & 15), g.items - 1), in, o, ts);
                const int r = dense_r(kk, lane);
                if (r > g.R - 1) T.ok = false;  // whole blocks stay inside the butterfly
                if (kk >= g.k4) continue;
                float2 xa = T.get(in + r * g.se), xb = T.get(in + (g.R - r) * g.se);
                if (g.Ns > 1) {
                    if (r * ts >= P.n || (g.R - r) * ts >= P.n) T.ok = false;
                    float2 wa = tw[r * ts], wb = tw[(g.R - r) * ts];
                    xa = cmul(xa, INV ? cconj(wa) : wa);
                    xb = cmul(xb, INV ? cconj(wb) : wb);
                }
                const float2 sm = cadd(xa, xb), d = csub(xa, xb);
                for (int row = 0; row < 16; ++row) {
                    const float2 w = coef[(mt * g.kb * kDenseBlock + kk) * 64 + (lane & ~15) + row];
                    auto& a = acc[row * 16 + (lane & 15)];
                    a[0] = (float)(a[0] + (double)w.x * sm.x);
                    a[1] = (float)(a[1] + (double)w.x * sm.y);
                    a[2] = (float)(a[2] + (double)w.y * d.x);
                    a[3] = (float)(a[3] + (double)w.y * d.y);
                }
            }
        }
        close_block();
        for (int lane = 0; lane < 64; ++lane) {
            const int b = nt * 16 + (lane & 15);
            int in, o, ts;
            dense_item<COLFAST, LOG2C>(g, std::min(b, g.items - 1), in, o, ts);
            for (int v = 0; v < 4; ++v) {
                const int q = dense_q(mt, lane, v);
                if (q > g.h || b >= g.items) continue;
                const auto& a = sum[(q - 16 * mt) * 16 + (lane & 15)];
                const float2 m = make_float2(a[0] + a[3], a[1] - a[2]);
                const float2 p = make_float2(a[0] - a[3], a[1] + a[2]);
                T.put(out, o + q * g.Ns * g.es, INV ? p : m);
                if (q > 0 && 2 * q != g.R) T.put(out, o + (g.R - q) * g.Ns * g.es, INV ? m : p);
            }
        }
    }
    for (int c = 0; c < ncols; ++c)
        for (int e = 0; e < P.n; ++e)
            if (T.writes[e * es + c * cs] != 1) T.ok = false;
    T.v = out;
}

template <bool COLFAST, int LOG2C, bool INV>
static double run(int n, int ncols) {
    Plan P{};
    if (!make_dense_plan(n, P)) return -1.0;
    const int es = COLFAST ? ncols : 1, cs = COLFAST ? 1 : n;
    std::vector<float2> tw(n);
    for (int q = 0; q < n; ++q)
        tw[q] = make_float2((float)std::cos(-2.0 * M_PI * q / n), (float)std::sin(-2.0 * M_PI * q / n));
    Tile T;
    T.v.resize((size_t)n * ncols);
    if ((int)T.v.size() > kDenseElems) return -2.0;
    T.writes.resize(T.v.size());
    srand(n * 17 + ncols);
    for (auto& x : T.v) x = make_float2(rand() / (float)RAND_MAX - 0.5f, rand() / (float)RAND_MAX - 0.5f);
    const std::vector<float2> in = T.v;
    for (int s = 0; s < P.nstages; ++s) {
        switch (P.radix[s]) {
#define REG(R) case R: emu_reg<R, COLFAST, LOG2C, INV>(T, P, s, ncols, es, cs, tw.data()); break;
            REG(2) REG(3) REG(4) REG(5) REG(6) REG(7) REG(8) REG(9) REG(10) REG(11) REG(12) REG(13) REG(14)
            REG(15) REG(16)
            default: emu_dense<COLFAST, LOG2C, INV>(T, P, s, ncols, es, cs, tw.data());
        }
    }
    if (!T.ok) return -3.0;
    double maxerr = 0.0, maxref = 0.0;
    for (int c = 0; c < ncols; c += 5)
        for (int k = 0; k < n; ++k) {
            std::complex<double> acc = 0.0;
            for (int e = 0; e < n; ++e) {
                const float2 x = in[e * es + c * cs];
                acc += std::complex<double>(x.x, x.y) *
                       std::polar(1.0, (INV ? 2.0 : -2.0) * M_PI * (double)((long)k * e % n) / n);
            }
            const float2 y = T.v[k * es + c * cs];
            maxerr = std::fmax(maxerr, std::abs(acc - std::complex<double>(y.x, y.y)));
            maxref = std::fmax(maxref, std::abs(acc));
        }
    return maxerr / maxref;
}

int main() {
    int bad = 0, lengths = 0;
    for (int n = 2; n <= kMaxDenseLen; ++n) {
        Plan P{};
        if (!make_dense_plan(n, P)) continue;
        // every plan's shape; the transforms themselves for the edges of the
        // radix tiles, every stage count and a spread of the others
        ++lengths;
        int prod = 1;
        for (int s = 0; s < P.nstages; ++s) prod *= P.radix[s];
        if (prod != n || P.nstages > 3) ++bad;
        const bool edge = n <= 40 || n == 47 || n == 61 || n == 62 || n == 64 || n == 67 || n == 127 || n == 131 ||
                          n == 164 || n == 205 || n == 211 || n == 232 || n == 243 || n == 250 || n == 251 ||
                          n == 254 || n == 255 || n == 256 || n == 257 || n == 258 || n == 289 || n == 306 ||
                          n == 323 || n == 361 || n == 391 || n == 502 || n == 510 || n == 511 || n == 512;
        if (!edge && n % 13 != 5) continue;
        const int rows = std::max(1, std::min(32, kDenseElems / n));
        double e[6];
        e[0] = n <= 256 ? run<true, 4, false>(n, 16) : run<true, 3, false>(n, 8);
        e[1] = n <= 256 ? run<true, 4, true>(n, 16) : run<true, 3, true>(n, 8);
        e[2] = run<false, 0, false>(n, rows);
        e[3] = run<false, 0, true>(n, rows);
        e[4] = run<false, 0, false>(n, std::max(1, rows / 4));
        e[5] = run<false, 0, true>(n, std::max(1, rows / 2));
        double worst = 0.0;
        bool ok = true;
        for (double x : e) {
            ok = ok && x >= 0.0;
            worst = std::fmax(worst, x);
        }
        ok = ok && worst < 2e-6;
        printf("n=%4d [%d %d %d] %.2e %s\n", n, P.radix[0], P.nstages > 1 ? P.radix[1] : 1,
               P.nstages > 2 ? P.radix[2] : 1, worst, ok ? "ok" : "FAIL");
        if (!ok) ++bad;
    }
    printf("%d lengths\n%s\n", lengths, bad ? "FAILED" : "ALL OK");
    return bad ? 1 : 0;
}
