// Transforms of lengths known only at run time, up to 512 with every prime
// factor up to 256, in two or three stages.
//
// The stages are those of fft_core.hpp (self-sorting Stockham), in place in
// one LDS tile: every thread reads its share of a stage into registers, a
// barrier, then writes the outputs.  A stage is one of
//   - a register radix, 2 ... 16: a thread holds whole butterflies;
//   - a dense radix R, 17 ... 256: the DFT matrix itself, on the matrix
//     cores (v_mfma_f32_16x16x4_f32).  With s_r = x_r + x_{R-r} and
//     d_r = x_r - x_{R-r}, r = 1 ... h = R / 2,
//       X_q = A_q -+ i B_q,  X_{R-q} = A_q +- i B_q  (forward / inverse)
//       A_q = x_0 + sum_r s_r cos(2 pi q r / R),  B_q = sum_r d_r sin(2 pi q r / R),
//     q = 0 ... h (even R: r = h pairs with itself and counts half), i.e. two
//     real (h + 1) x h matrices times the real and imaginary parts of the
//     tile's butterflies.  One wave computes a unit of 16 rows q by 16
//     butterflies: 16 accumulator registers, h / 4 steps of four MFMAs.
//
// Why: a length with a prime factor p > 13 ran as a chirp-z transform, two
// convolution transforms of length M >= 2n - 1 with three passes over the
// tile around them and two LDS buffers of M rows (one or two blocks per CU).
// A dense radix costs R - 1 multiply-adds per element, which at the 128 per
// clock and CU of the FP32 MFMA is below the time the pass needs for HBM up
// to about R = 200, and the tile stays at n rows.
#pragma once

#include "fft_col2.hpp"

namespace qsmfft {

constexpr int kMaxDenseLen = 512;    // tiles of 16 columns up to 256, 8 above
constexpr int kMaxDenseRadix = 256;  // above, only primes: chirp-z (fft_chirp.hpp)
constexpr int kMaxRegRadix = 16;
constexpr int kDenseElems = 16 * kThreads;  // elements of the largest tile
constexpr int kDenseUnits = 4;              // units one wave holds (16 accumulators each)

template <bool INV> struct Dft<6, INV> : DftSplit<2, 3, INV> {};

__host__ __device__ constexpr int dense_row_tiles(int R) { return (R / 2 + 16) / 16; }  // of the h + 1 rows
__host__ __device__ constexpr int dense_k_steps(int R) { return (R / 2 + 3) / 4; }
// float2 entries of a dense radix's coefficient table
__host__ __device__ constexpr int dense_table_len(int R) { return dense_row_tiles(R) * dense_k_steps(R) * 64; }

// Geometry of one dense stage over a tile.
struct DenseGeom {
    int R, h, mt, k4;    // rows 0 ... h in mt tiles of 16, k4 steps of four r
    int items, units;    // butterflies of the tile; (item tile, row tile) pairs
    int nb, Ns, tstep;   // as StageGeom
    int es, cs, se;      // element and sequence strides, input stride nb * es
    uint64_t m_nb, m_Ns;
};
__host__ __device__ __forceinline__ DenseGeom dense_geom(const Plan& P, int s, int ncols, int es, int cs) {
    DenseGeom g;
    g.R = P.radix[s];
    g.h = g.R / 2;
    g.mt = dense_row_tiles(g.R);
    g.k4 = dense_k_steps(g.R);
    g.nb = P.n / g.R;
    g.Ns = P.ns[s];
    g.tstep = g.nb / g.Ns;
    g.items = g.nb * ncols;
    g.units = ((g.items + 15) >> 4) * g.mt;
    g.es = es;
    g.cs = cs;
    g.se = g.nb * es;
    g.m_nb = P.m_nb[s];
    g.m_Ns = P.m_ns[s];
    return g;
}
// Butterfly b (clamped to the tile's by the caller) of a dense stage: the LDS
// index of its input 0, the LDS index of its output 0, and its twiddle step.
template <bool COLFAST, int LOG2C>
__host__ __device__ __forceinline__ void dense_item(const DenseGeom& g, int b, int& in, int& out, int& ts) {
    int j, c;
    if (COLFAST) {
        c = b & ((1 << LOG2C) - 1);
        j = b >> LOG2C;
    } else {
        c = (int)fastdiv((uint32_t)b, g.m_nb);
        j = b - c * g.nb;
    }
    const int grp = (int)fastdiv((uint32_t)j, g.m_Ns);
    const int k = j - grp * g.Ns;
    in = j * g.es + c * g.cs;
    out = (grp * g.Ns * g.R + k) * g.es + c * g.cs;
    ts = k * g.tstep;
}
// Lane roles of a unit: operands of step kk at r = dense_r, results v = 0..3
// at row q = dense_q, item (lane & 15) of the unit's item tile.
__host__ __device__ __forceinline__ int dense_r(int kk, int lane) { return 4 * kk + (lane >> 4) + 1; }
__host__ __device__ __forceinline__ int dense_q(int mt, int lane, int v) { return 16 * mt + 4 * (lane >> 4) + v; }

// Register-radix stage in place, as fixed_stage_load / _store with run-time
// geometry: B butterflies per thread at most.
template <int R>
struct RegStage {
    static constexpr int B = (kDenseElems / kThreads + R - 1) / R;
};
template <int R, bool COLFAST, int LOG2C>
__host__ __device__ __forceinline__ void reg_stage_load(const float2* lds, int tid, const StageGeom& g,
                                                        float2 (&v)[RegStage<R>::B][R]) {
    const int total = g.nb * g.ncols;
#pragma unroll
    for (int t = 0; t < RegStage<R>::B; ++t) {
        const int b = tid + t * kThreads;
        if (b < total) {
            int j, c;
            split_b<COLFAST, LOG2C>(b, g, j, c);
            const float2* p = lds + j * g.es + c * g.cs;
#pragma unroll
            for (int r = 0; r < R; ++r) v[t][r] = p[r * g.nb * g.es];
        }
    }
}
template <int R, bool COLFAST, int LOG2C, bool INV>
__host__ __device__ __forceinline__ void reg_stage_store(float2* lds, int tid, const StageGeom& g,
                                                         float2 (&v)[RegStage<R>::B][R], const float2* tw) {
    const int total = g.nb * g.ncols;
#pragma unroll
    for (int t = 0; t < RegStage<R>::B; ++t) {
        const int b = tid + t * kThreads;
        if (b < total) {
            int j, c;
            split_b<COLFAST, LOG2C>(b, g, j, c);
            const int grp = (int)fastdiv((uint32_t)j, g.m_Ns);
            const int k = j - grp * g.Ns;
            if (g.Ns > 1) {
                const int ts = k * g.tstep;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    float2 w = tw[r * ts];
                    if (INV) w = cconj(w);
                    v[t][r] = cmul(v[t][r], w);
                }
            }
            Dft<R, INV>::run(v[t], tw, g.n);
            float2* q = lds + (grp * g.Ns * R + k) * g.es + c * g.cs;
#pragma unroll
            for (int r = 0; r < R; ++r) q[r * g.Ns * g.es] = v[t][r];
        }
    }
}

#ifdef __HIPCC__
typedef float mfma_f4 __attribute__((ext_vector_type(4)));

// One dense stage on the device.  coef: the radix's table in global memory,
// entry (mt, kk, lane) = (cos, sin)(2 pi q r / R) for the row q = 16 mt +
// (lane & 15) and the r of dense_r (zero past either end).  All lanes of a
// wave take part in every MFMA; items past the tile's last repeat it and are
// not written.  Barriers: the caller's before, one between the reads and the
// writes, one after.
template <bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ void dense_stage(float2* lds, const DenseGeom& g, const float2* tw,
                                            const float2* __restrict__ coef) {
    const int lane = (int)(threadIdx.x & 63);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    mfma_f4 are[kDenseUnits], aim[kDenseUnits], bre[kDenseUnits], bim[kDenseUnits];
#pragma unroll
    for (int u = 0; u < kDenseUnits; ++u) {
        const int unit = wv + u * (kThreads / 64);
        if (unit < g.units) {
            const int nt = unit / g.mt, mt = unit - nt * g.mt;
            int in, out, ts;
            dense_item<COLFAST, LOG2C>(g, min(nt * 16 + (lane & 15), g.items - 1), in, out, ts);
            const float2 x0 = lds[in];
            mfma_f4 ar = {x0.x, x0.x, x0.x, x0.x}, ai = {x0.y, x0.y, x0.y, x0.y};
            mfma_f4 br = {0.0f, 0.0f, 0.0f, 0.0f}, bi = {0.0f, 0.0f, 0.0f, 0.0f};
            const float2* __restrict__ cf = coef + mt * g.k4 * 64 + lane;
            float2 w = *cf;
            for (int kk = 0; kk < g.k4; ++kk) {
                const int r = min(dense_r(kk, lane), g.h);  // (coefficients are 0 past h)
                float2 xa = lds[in + r * g.se], xb = lds[in + (g.R - r) * g.se];
                cf += 64;
                const float2 wn = kk + 1 < g.k4 ? *cf : w;  // the next step's, in flight
                if (g.Ns > 1) {
                    float2 wa = tw[r * ts], wb = tw[(g.R - r) * ts];
                    if (INV) {
                        wa = cconj(wa);
                        wb = cconj(wb);
                    }
                    xa = cmul(xa, wa);
                    xb = cmul(xb, wb);
                }
                const float2 s = cadd(xa, xb), d = csub(xa, xb);
                ar = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, s.x, ar, 0, 0, 0);
                ai = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, s.y, ai, 0, 0, 0);
                br = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, d.x, br, 0, 0, 0);
                bi = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, d.y, bi, 0, 0, 0);
                w = wn;
            }
            are[u] = ar;
            aim[u] = ai;
            bre[u] = br;
            bim[u] = bi;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kDenseUnits; ++u) {
        const int unit = wv + u * (kThreads / 64);
        if (unit < g.units) {
            const int nt = unit / g.mt, mt = unit - nt * g.mt;
            const int b = nt * 16 + (lane & 15);
            int in, out, ts;
            dense_item<COLFAST, LOG2C>(g, min(b, g.items - 1), in, out, ts);
            const int so = g.Ns * g.es;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int q = dense_q(mt, lane, v);
                if (q <= g.h && b < g.items) {
                    const float2 m = make_float2(are[u][v] + bim[u][v], aim[u][v] - bre[u][v]);  // A - i B
                    const float2 p = make_float2(are[u][v] - bim[u][v], aim[u][v] + bre[u][v]);  // A + i B
                    lds[out + q * so] = INV ? p : m;
                    if (q > 0 && 2 * q != g.R) lds[out + (g.R - q) * so] = INV ? m : p;
                }
            }
        }
    }
    __syncthreads();
}

template <int R, bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ void reg_stage(float2* lds, const Plan& P, int s, int ncols, int es, int cs,
                                          const float2* tw) {
    const StageGeom g = plan_geom(P, s, ncols, es, cs);
    float2 v[RegStage<R>::B][R];
    reg_stage_load<R, COLFAST, LOG2C>(lds, threadIdx.x, g, v);
    __syncthreads();
    reg_stage_store<R, COLFAST, LOG2C, INV>(lds, threadIdx.x, g, v, tw);
    __syncthreads();
}

// Full transform, in place in lds (ncols sequences of P.n elements at
// e * es + c * cs).  tw: the twiddle table in LDS; twg: the bank in global
// memory (the dense tables).  The caller has synchronised after filling the
// tile; returns after a final barrier.
template <bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ void lds_fft_dense(float2* lds, const Plan& P, int ncols, int es, int cs,
                                              const float2* tw, const float2* __restrict__ twg) {
    for (int s = 0; s < P.nstages; ++s) {
        switch (P.radix[s]) {
            case 2: reg_stage<2, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 3: reg_stage<3, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 4: reg_stage<4, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 5: reg_stage<5, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 6: reg_stage<6, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 7: reg_stage<7, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 8: reg_stage<8, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 9: reg_stage<9, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 10: reg_stage<10, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 11: reg_stage<11, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 12: reg_stage<12, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 13: reg_stage<13, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 14: reg_stage<14, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 15: reg_stage<15, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 16: reg_stage<16, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            default: dense_stage<COLFAST, LOG2C, INV>(lds, dense_geom(P, s, ncols, es, cs), tw, twg + P.dn_off[s]);
        }
    }
}
#endif

// --------------------------------------------------------- host planning --
// Cost of a stage per element, in clocks of one CU: the LDS round trip and
// its barriers, and for a dense radix its MFMAs (2 mt k4 / R).
inline double dense_stage_cost(int R) {
    if (R <= kMaxRegRadix) return 0.55 + 0.004 * R;
    return 0.45 + 2.0 * dense_row_tiles(R) * dense_k_steps(R) / R;
}

// The cheapest ordered split of n into at most three stages, dense radices
// first (the first stage has no twiddles).  False where n has a prime factor
// above kMaxDenseRadix or is above kMaxDenseLen.
inline bool dense_factorize(int n, int* radix, int* nstages) {
    if (n < 1 || n > kMaxDenseLen) return false;
    if (n == 1) {
        *nstages = 0;
        return true;
    }
    double best = 0.0;
    *nstages = 0;
    auto offer = [&](int a, int b, int c) {
        double cost = dense_stage_cost(a);
        if (b > 1) cost += dense_stage_cost(b);
        if (c > 1) cost += dense_stage_cost(c);
        if (*nstages && cost >= best) return;
        best = cost;
        *nstages = 1 + (b > 1) + (c > 1);
        radix[0] = a;
        radix[1] = b;
        radix[2] = c;
    };
    for (int a = 2; a <= n && a <= kMaxDenseRadix; ++a) {
        if (n % a) continue;
        const int m = n / a;
        for (int b = 1; b <= a && b <= m; ++b) {
            if (m % b) continue;
            const int c = m / b;
            if (c <= b || b == 1) {
                if (b == 1 && c != 1) continue;
                offer(a, b, c);
            }
        }
    }
    return *nstages > 0;
}

// Fill a plan for length n (dn_off is left to the caller).
inline bool make_dense_plan(int n, Plan& p) {
    p.n = n;
    if (!dense_factorize(n, p.radix, &p.nstages)) return false;
    int ns = 1;
    for (int s = 0; s < p.nstages; ++s) {
        p.ns[s] = ns;
        p.m_nb[s] = magic_for((uint32_t)(n / p.radix[s]));
        p.m_ns[s] = magic_for((uint32_t)ns);
        ns *= p.radix[s];
    }
    p.dense = 1;
    return true;
}

// Coefficient table of a dense radix (see dense_stage), from exactly reduced
// angles in long double.  Even R: r = h is its own pair, so its sum counts it
// twice and its cosine is halved (its difference is 0).
inline void dense_table(int R, float2* out) {
    const long double two_pi = 6.283185307179586476925286766559L;
    const int h = R / 2;
    for (int mt = 0; mt < dense_row_tiles(R); ++mt)
        for (int kk = 0; kk < dense_k_steps(R); ++kk)
            for (int lane = 0; lane < 64; ++lane) {
                const int q = 16 * mt + (lane & 15), r = dense_r(kk, lane);
                float2 w = make_float2(0.0f, 0.0f);
                if (q <= h && r <= h) {
                    const long double a = two_pi * ((q * r) % R) / R;
                    const long double half = 2 * r == R ? 0.5L : 1.0L;
                    w = make_float2((float)(half * cosl(a)), 2 * r == R ? 0.0f : (float)sinl(a));
                }
                out[(mt * dense_k_steps(R) + kk) * 64 + lane] = w;
            }
}

}  // namespace qsmfft
