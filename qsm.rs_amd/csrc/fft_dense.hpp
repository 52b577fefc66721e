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

#include <cmath>

#include "fft_col2.hpp"

namespace qsmfft {

constexpr int kMaxDenseLen = 512;    // tiles of 16 columns up to 256, 8 above
constexpr int kMaxDenseRadix = 256;  // above, only primes: chirp-z (fft_chirp.hpp)
constexpr int kMaxRegRadix = 16;
constexpr int kDenseElems = 16 * kThreads;  // elements of the largest tile
constexpr int kDenseUnits = 4;              // units one wave holds (16 accumulators each) of such a tile

template <bool INV> struct Dft<6, INV> : DftSplit<2, 3, INV> {};

__host__ __device__ constexpr int dense_row_tiles(int R) { return (R / 2 + 16) / 16; }  // of the h + 1 rows
__host__ __device__ constexpr int dense_k_steps(int R) { return (R / 2 + 3) / 4; }
// MFMA steps (of four r) summed before they join the total, whose operands
// are loaded together: in one chain the error grows with R, 1.9e-7 at 211
// points against the chirp-z transform's 1.5e-7 (relative, random input); in
// blocks of 16 r it stays at 1.0e-7.
constexpr int kDenseBlock = 4;
// blocks of a radix, and float2 entries of its coefficient table (whole blocks)
__host__ __device__ constexpr int dense_blocks(int R) { return (dense_k_steps(R) + kDenseBlock - 1) / kDenseBlock; }
__host__ __device__ constexpr int dense_table_len(int R) {
    return dense_row_tiles(R) * dense_blocks(R) * kDenseBlock * 64;
}

// Geometry of one dense stage over a tile.
struct DenseGeom {
    int R, h, mt, k4;    // rows 0 ... h in mt tiles of 16, k4 steps of four r
    int kb;              // blocks of kDenseBlock steps
    int items, units;    // butterflies of the tile; (item tile, row tile) pairs
    int m_mt;            // ceil(2^16 / mt): unit / mt = unit * m_mt >> 16
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
    g.kb = dense_blocks(g.R);
    g.nb = P.nb[s];
    g.Ns = P.ns[s];
    g.tstep = P.tst[s];
    g.items = g.nb * ncols;
    g.units = ((g.items + 15) >> 4) * g.mt;
    g.m_mt = (65536 + g.mt - 1) / g.mt;
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
// Item tile and row tile of a unit (unit < 32).
__host__ __device__ __forceinline__ void dense_unit(const DenseGeom& g, int unit, int& nt, int& mt) {
    nt = (unit * g.m_mt) >> 16;
    mt = unit - nt * g.mt;
}
// Lane roles of a unit: operands of step kk at r = dense_r, results v = 0..3
// at row q = dense_q, item (lane & 15) of the unit's item tile.
__host__ __device__ __forceinline__ int dense_r(int kk, int lane) { return 4 * kk + (lane >> 4) + 1; }
__host__ __device__ __forceinline__ int dense_q(int mt, int lane, int v) { return 16 * mt + 4 * (lane >> 4) + v; }

// Register-radix stage in place, as fixed_stage_load / _store with run-time
// geometry: B butterflies per thread at most, in a tile of E elements per
// thread (16, or 8: half tiles).
template <int R, int E = kDenseElems / kThreads>
struct RegStage {
    static constexpr int B = (E + R - 1) / R;
};
template <int R, bool COLFAST, int LOG2C, int E = kDenseElems / kThreads>
__host__ __device__ __forceinline__ void reg_stage_load(const float2* lds, int tid, const StageGeom& g,
                                                        float2 (&v)[RegStage<R, E>::B][R]) {
    const int total = g.nb * g.ncols;
#pragma unroll
    for (int t = 0; t < RegStage<R, E>::B; ++t) {
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
template <int R, bool COLFAST, int LOG2C, bool INV, int E = kDenseElems / kThreads>
__host__ __device__ __forceinline__ void reg_stage_store(float2* lds, int tid, const StageGeom& g,
                                                         float2 (&v)[RegStage<R, E>::B][R], const float2* tw) {
    const int total = g.nb * g.ncols;
#pragma unroll
    for (int t = 0; t < RegStage<R, E>::B; ++t) {
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
// not written.  A block's coefficients are fetched one block ahead (the next
// unit's included): fetched a step ahead they held each step for an L2 round
// trip.  Barriers: the caller's before, one between the reads and the writes,
// one after.
template <int E, bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ void dense_stage(float2* lds, const DenseGeom& g, const float2* tw,
                                            const float2* __restrict__ coef) {
    const int lane = (int)(threadIdx.x & 63);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int bstep = kDenseBlock * 64;
    constexpr int UNITS = kDenseUnits * E * kThreads / kDenseElems;
    mfma_f4 are[UNITS], aim[UNITS], bre[UNITS], bim[UNITS];
    const mfma_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float2 w[kDenseBlock];
    auto fetch = [&](int unit, int kb) {  // in bounds for every unit (mt < g.mt) and kb < g.kb
        int nt, mt;
        dense_unit(g, unit, nt, mt);
        const float2* __restrict__ cf = coef + (mt * g.kb + kb) * bstep;
#pragma unroll
        for (int t = 0; t < kDenseBlock; ++t) w[t] = (cf + t * 64)[(unsigned)lane];
    };
    fetch(wv, 0);
    const int se4 = 4 * g.se;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int unit = wv + u * (kThreads / 64);
        if (unit < g.units) {
            int nt, mt, in, out, ts;
            dense_unit(g, unit, nt, mt);
            dense_item<COLFAST, LOG2C>(g, min(nt * 16 + (lane & 15), g.items - 1), in, out, ts);
            const float2 x0 = lds[in];
            are[u] = mfma_f4{x0.x, x0.x, x0.x, x0.x};
            aim[u] = mfma_f4{x0.y, x0.y, x0.y, x0.y};
            bre[u] = bim[u] = zero;
            // inputs r and R - r of step 0, stepped by 4; past h (where the
            // coefficients are 0) they stay inside the butterfly: a whole
            // block ends at r <= R - 1 for every R >= 17
            const int r0 = dense_r(0, lane);
            const float2* pa = lds + in + r0 * g.se;
            const float2* pb = lds + in + (g.R - r0) * g.se;
            const float2* ta = tw + r0 * ts;
            const float2* tb = tw + (g.R - r0) * ts;
            for (int kb = 0; kb < g.kb; ++kb) {
                float2 xa[kDenseBlock], xb[kDenseBlock], wc[kDenseBlock];
#pragma unroll
                for (int t = 0; t < kDenseBlock; ++t) {
                    xa[t] = *pa;
                    xb[t] = *pb;
                    pa += se4;
                    pb -= se4;
                    if (g.Ns > 1) {
                        float2 wa = *ta, wb = *tb;
                        ta += 4 * ts;
                        tb -= 4 * ts;
                        if (INV) {
                            wa = cconj(wa);
                            wb = cconj(wb);
                        }
                        xa[t] = cmul(xa[t], wa);
                        xb[t] = cmul(xb[t], wb);
                    }
                    wc[t] = w[t];
                }
                if (kb + 1 < g.kb) fetch(unit, kb + 1);
                else fetch(unit + kThreads / 64, 0);
                mfma_f4 ar = zero, ai = zero, br = zero, bi = zero;
#pragma unroll
                for (int t = 0; t < kDenseBlock; ++t) {
                    if (t == 0 || kb * kDenseBlock + t < g.k4) {
                        const float2 s = cadd(xa[t], xb[t]), d = csub(xa[t], xb[t]);
                        ar = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[t].x, s.x, ar, 0, 0, 0);
                        ai = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[t].x, s.y, ai, 0, 0, 0);
                        br = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[t].y, d.x, br, 0, 0, 0);
                        bi = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[t].y, d.y, bi, 0, 0, 0);
                    }
                }
                are[u] += ar;
                aim[u] += ai;
                bre[u] += br;
                bim[u] += bi;
            }
        }
    }
    __syncthreads();
    const int so = g.Ns * g.es;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int unit = wv + u * (kThreads / 64);
        if (unit < g.units) {
            int nt, mt, in, out, ts;
            dense_unit(g, unit, nt, mt);
            const int b = nt * 16 + (lane & 15);
            dense_item<COLFAST, LOG2C>(g, min(b, g.items - 1), in, out, ts);
            const int q0 = dense_q(mt, lane, 0);
            float2* oq = lds + out + q0 * so;
            float2* om = lds + out + (g.R - q0) * so;
            const int hv = b < g.items ? g.h : -1;  // (items past the last write nothing)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int q = q0 + v;
                const float2 m = make_float2(are[u][v] + bim[u][v], aim[u][v] - bre[u][v]);  // A - i B
                const float2 p = make_float2(are[u][v] - bim[u][v], aim[u][v] + bre[u][v]);  // A + i B
                if (q <= hv) *oq = INV ? p : m;
                if (q <= hv && q > 0 && 2 * q != g.R) *om = INV ? m : p;
                oq += so;
                om -= so;
            }
        }
    }
    __syncthreads();
}

template <int R, int E, bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ void reg_stage(float2* lds, const Plan& P, int s, int ncols, int es, int cs,
                                          const float2* tw) {
    const StageGeom g = plan_geom(P, s, ncols, es, cs);
    float2 v[RegStage<R, E>::B][R];
    reg_stage_load<R, COLFAST, LOG2C, E>(lds, threadIdx.x, g, v);
    __syncthreads();
    reg_stage_store<R, COLFAST, LOG2C, INV, E>(lds, threadIdx.x, g, v, tw);
    __syncthreads();
}

// Full transform, in place in lds (ncols sequences of P.n elements at
// e * es + c * cs).  tw: the twiddle table in LDS; twg: the bank in global
// memory (the dense tables); E: the tile's elements per thread.  The caller has
// synchronised after filling the tile; returns after a final barrier.
template <int E, bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ void lds_fft_dense(float2* lds, const Plan& P, int ncols, int es, int cs,
                                              const float2* tw, const float2* __restrict__ twg) {
    for (int s = 0; s < P.nstages; ++s) {
        switch (P.radix[s]) {
            case 2: reg_stage<2, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 3: reg_stage<3, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 4: reg_stage<4, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 5: reg_stage<5, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 6: reg_stage<6, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 7: reg_stage<7, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 8: reg_stage<8, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 9: reg_stage<9, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 10: reg_stage<10, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 11: reg_stage<11, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 12: reg_stage<12, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 13: reg_stage<13, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 14: reg_stage<14, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 15: reg_stage<15, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            case 16: reg_stage<16, E, COLFAST, LOG2C, INV>(lds, P, s, ncols, es, cs, tw); break;
            default: dense_stage<E, COLFAST, LOG2C, INV>(lds, dense_geom(P, s, ncols, es, cs), tw, twg + P.dn_off[s]);
        }
    }
}
#endif

// --------------------------------------------------------- host planning --
// Cost of a stage per element, in clocks of one CU: the LDS round trip and
// its barriers, and for a dense radix its MFMAs (2 mt k4 / R).  0: no such
// stage.  A dense radix has a prime factor above 13: where register radices
// suffice their fewer roundings are kept (at 40 points 1.2e-7 of the largest
// output against 1.7e-7 for the dense matrix).
inline double dense_stage_cost(int R) {
    if (R <= kMaxRegRadix) return 0.55 + 0.004 * R;
    int m = R;
    for (int p : {2, 3, 5, 7, 11, 13})
        while (m % p == 0) m /= p;
    if (m == 1 || R > kMaxDenseRadix) return 0.0;
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
        const double ca = dense_stage_cost(a), cb = b > 1 ? dense_stage_cost(b) : 0.0,
                     cc = c > 1 ? dense_stage_cost(c) : 0.0, cost = ca + cb + cc;
        if (ca == 0.0 || (b > 1 && cb == 0.0) || (c > 1 && cc == 0.0)) return;
        if (*nstages && cost >= best) return;
        best = cost;
        *nstages = 1 + (b > 1) + (c > 1);
        radix[0] = a;
        radix[1] = b;
        radix[2] = c;
    };
    for (int a = 2; a <= n; ++a) {
        if (n % a) continue;
        const int m = n / a;
        for (int b = 1; b <= a && b <= m; ++b)
            if (m % b == 0 && m / b <= b) offer(a, b, m / b);  // a >= b >= c
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
        p.nb[s] = n / p.radix[s];
        p.tst[s] = n / (ns * p.radix[s]);
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
    float2 root[kMaxDenseRadix];
    for (int m = 0; m < R; ++m) {
        const long double a = two_pi * m / R;
        root[m] = make_float2((float)cosl(a), (float)sinl(a));
    }
    for (int mt = 0; mt < dense_row_tiles(R); ++mt)
        for (int kk = 0; kk < dense_blocks(R) * kDenseBlock; ++kk)
            for (int lane = 0; lane < 64; ++lane) {
                const int q = 16 * mt + (lane & 15), r = dense_r(kk, lane);
                float2 w = make_float2(0.0f, 0.0f);
                if (q <= h && r <= h) {
                    w = root[(q * r) % R];
                    if (2 * r == R) w = make_float2(0.5f * w.x, 0.0f);
                }
                out[(mt * dense_blocks(R) * kDenseBlock + kk) * 64 + lane] = w;
            }
}

}  // namespace qsmfft
