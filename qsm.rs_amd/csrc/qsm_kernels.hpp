// Pass kernels of the TV-ADMM and V-SHARP paths, as templates on the length
// N of the transformed axis (N = 0: runtime plan with EG elements per thread).
//
// The 3-D transforms are real-to-complex along x (two real rows packed as one
// complex row), then complex along y and z on the half spectrum, in three
// LDS-staged passes; element-wise work is fused into the passes:
//   TV-ADMM iteration (src/inversion/admm.rs:76-145):
//     k_r2c_x<TVDIV>   z/u update of the previous iteration + bdiv + R2C x
//     k_y_pass<fwd>    C2C along y
//     k_z_tv<SOLVE>    C2C z, x^ = f^ - rho*inv_a*FFT(div), inverse z
//     k_y_pass<inv>    inverse C2C along y
//     k_c2r_tv         C2R x, write x, partial sums of relative_change
//   V-SHARP radius (src/bgremove/vsharp.rs:132-177):
//     k_r2c_x<SPHERE>, k_y_pass<fwd>, k_z_vs<RADIUS>, k_y_pass<inv> (x2),
//     k_c2r_vs_select
// Global phases issue all of a thread's loads before the first wait (loops
// over a compile-time count into registers); twiddles are staged in LDS.
#pragma once

#include <type_traits>

#include "fft_dense.hpp"
#include "qsm_internal.hpp"

namespace qsm {

using qsmfft::kThreads;
using qsmfft::fastdiv;

constexpr int kMaxLen = 1024;

// Device pointers held in the volume descriptor are generic (flat) to the
// compiler; accessed through global-address-space types they compile to
// global loads/stores with a scalar base instead of flat operations, which
// also keeps them off the LDS wait counter.
#define QSM_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ QSM_GLOBAL T* glb(T* p) { return (QSM_GLOBAL T*)p; }
template <class T>
__device__ __forceinline__ const QSM_GLOBAL T* glb(const T* p) { return (const QSM_GLOBAL T*)p; }

// 8-byte complex access through a global pointer (one dwordx2 load/store).
typedef float qsm_f2v __attribute__((ext_vector_type(2)));
// One load / store, NT: with the non-temporal hint (first out of the caches).
//
// The TV iteration's passes come in an NT form for batches whose arrays (40
// bytes a voxel: x and u twice, two spectra) are larger than the 256 MB
// Infinity Cache (kStreamBytes; the host chooses).  Without a hint each array
// evicts the next and nothing is left when it is read again; with it the dual
// variable and f^, read again only an iteration later, and the spectrum's last
// reading leave the cache to the spectrum and x, which the next pass reads.
// Measured, us an iteration without and with: two 384x384x256 volumes (3.0
// GB) 1085 and 1061 (the z pass 170 and 143), four 256x256x160 (1.7 GB) 545
// and 526, one 250x250x200 (500 MB) 286 and 270, one 256x256x160 (419 MB) 155
// and 154, one 256x256x144 (377 MB) 144 and 144.  Where it fits the hint
// loses: 224x224x128 (257 MB) 101 and 104, 192x192x128 (189 MB) 78 and 86.
template <bool NT, class T>
__device__ __forceinline__ T ldx(const QSM_GLOBAL T* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT, class T>
__device__ __forceinline__ void stx(QSM_GLOBAL T* p, T v) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}
template <bool NT = false>
__device__ __forceinline__ float2 ldg2(const QSM_GLOBAL float2* p) {
    const qsm_f2v v = ldx<NT>((const QSM_GLOBAL qsm_f2v*)p);
    return make_float2(v.x, v.y);
}
__device__ __forceinline__ void stg2(QSM_GLOBAL float2* p, float2 a) {
    qsm_f2v v;
    v.x = a.x;
    v.y = a.y;
    *(QSM_GLOBAL qsm_f2v*)p = v;
}

// elements per thread of an x (row) pass / a column pass, LDS tile sizes and
// twiddle entries (n: compiled length or 0; eg: a run-time kernel's EG)
__host__ __device__ constexpr int x_emax(int n, int eg) {
    return n > 0 ? (qsmfft::fixed_rows(n) * n + kThreads - 1) / kThreads : (eg_dense(eg) ? eg_elems(eg) : kRowEmaxRt);
}
__host__ __device__ constexpr int col_emax(int n, int eg) {
    return n > 0 ? (kTile * n + kThreads - 1) / kThreads : eg_elems(eg);
}
__host__ __device__ constexpr int x_lds(int n, int eg) {
    return n > 0 ? qsmfft::fixed_rows(n) * n : kThreads * x_emax(n, eg);
}
__host__ __device__ constexpr int col_lds(int n, int eg) { return n > 0 ? kTile * n : kThreads * eg_elems(eg); }
__host__ __device__ constexpr int tw_lds(int n, int eg) {
    return n > 0 ? n : (eg_dense(eg) ? qsmfft::kMaxDenseLen : kMaxLen);
}
// column passes of the lengths fft_col2.hpp covers use its padded layout
__host__ __device__ constexpr int col_lds2(int n, int eg) {
    return qsmfft::col2_ok(n) ? 16 * n + 256 : col_lds(n, eg);
}

// The second LDS buffer of the runtime-plan transforms: one per kernel and
// size, shared by every transform the kernel runs.
template <int SIZE>
__device__ __forceinline__ float2* pp_buffer() {
    __shared__ float2 pp[SIZE];
    return pp;
}

// The transform of a runtime plan of work length 1024 (a chirp-z convolution,
// or that length itself) on the compile-time stages (fft_fixed.hpp), in place
// in buf, when the tile holds the sequences those stages are built for:
// column tiles of 2^LOG2C columns (layout e * 2^LOG2C + c), or row tiles of
// kThreads * EMAX / 1024 sequences at stride 1024.  Returns false (nothing
// done) otherwise.
template <int EMAX, bool COLFAST, int LOG2C, bool INV>
__device__ __forceinline__ bool fixed_1024_stages(float2* buf, const qsmfft::Plan& P, int ncols, const float2* twl) {
    constexpr int M = 1024, NC = COLFAST ? (1 << LOG2C) : (kThreads * EMAX) / M;
    if (P.n != M || ncols != NC) return false;
    qsmfft::fixed_fft<M, NC, COLFAST, INV>(buf, twl);
    return true;
}

// twl: the pass's twiddle table in LDS; twg: the twiddle bank in global
// memory (the chirp-z tables of runtime-planned lengths).
template <int N, int EG, int EMAX, bool COLFAST, int LOG2C, bool INV, int NC = 0>
__device__ __forceinline__ void run_fft(float2* lds, const qsmfft::Plan& P, int ncols, int es, int cs,
                                        const float2* twl, const float2* twg) {
    if constexpr (N > 0) {
        qsmfft::fixed_fft<N, NC ? NC : (COLFAST ? kTile : qsmfft::fixed_rows(N)), COLFAST, INV>(lds, twl);
    } else if constexpr (eg_dense(EG)) {
        qsmfft::lds_fft_dense<EMAX, COLFAST, LOG2C, INV>(lds, P, ncols, es, cs, twl, twg);
    } else {
        // runtime-planned lengths (513 ... 1024, and chirp-z primes above 256):
        // out-of-place stages between the kernel's tile (kThreads * EMAX
        // elements in every such kernel) and a second buffer of that size
        auto inner = [&](float2* src, float2* dst, auto inv, int wes, int wcs) -> float2* {
            constexpr bool I = decltype(inv)::value;
            if (fixed_1024_stages<EMAX, COLFAST, LOG2C, I>(src, P, ncols, twl)) return src;
            return qsmfft::plan_stages<COLFAST, LOG2C, I>(src, dst, P, ncols, wes, wcs, twl);
        };
        qsmfft::lds_fft_any<COLFAST, LOG2C, INV>(lds, pp_buffer<kThreads * EMAX>(), P, ncols, es, cs, twg, inner);
    }
}

// A pass's twiddle table (exp(-2 pi i q / n), q < n) is fetched into
// registers before the pass issues its tile loads and written to LDS after
// them: a table load whose value had to reach LDS first would hold every block
// for one memory round trip before its tile loads went out.
// The table of plan P (its length P.n: the axis length, or the chirp-z
// convolution length).
template <int N, int EG = 0>
struct TwStage {
    static constexpr int K = (tw_lds(N, EG) + kThreads - 1) / kThreads;
    float2 r[K];
    int n;
    __device__ __forceinline__ void fetch(const float2* __restrict__ tw, const qsmfft::Plan& P) {
        n = N > 0 ? N : P.n;
        const QSM_GLOBAL float2* g = glb(tw + P.tw_off);
#pragma unroll
        for (int t = 0; t < K; ++t) r[t] = ldg2(g + min((int)threadIdx.x + t * kThreads, n - 1));
    }
    // threads past n hold entry n - 1 and write it again (no branch)
    __device__ __forceinline__ void commit(float2* twl) const {
#pragma unroll
        for (int t = 0; t < K; ++t) twl[min((int)threadIdx.x + t * kThreads, n - 1)] = r[t];
    }
};

// exp(-2 pi i k / n) of a z pass: its twiddle table, except for a chirp-z
// length, whose table is that of the convolution length.
template <int N>
__device__ __forceinline__ float2 ztw(const VolDesc& V, const float2* twl, int kz, int nz) {
    if (N == 0 && V.pz.bl_n) {
        float sn, cs;
        sincospif(-2.0f * (float)kz / (float)nz, &sn, &cs);
        return make_float2(cs, sn);
    }
    return twl[kz];
}

// e / nx and e / nxh for an element of a row tile (e < 2^16)
template <int N>
__device__ __forceinline__ int div_nx(int e, const VolDesc& V) {
    if constexpr (N > 0) return e / N;
    else return (int)fastdiv((uint32_t)e, V.m_nx);
}
template <int N>
__device__ __forceinline__ int div_nxh(int e, const VolDesc& V) {
    if constexpr (N > 0) return e / ((N + 1) / 2);
    else return (int)fastdiv((uint32_t)e, V.m_nxh);
}

__device__ __forceinline__ float shrinkf(float x, float t) {
    // src/utils/mod.rs:44-52
    return x > t ? x - t : (x < -t ? x + t : 0.0f);
}

__device__ inline double block_sum(double v, double* sh) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / 64; ++w) s += sh[w];
    return s;
}

// relative_change = ||x - x_prev|| / (||x|| + 1e-20), converged when < tol
// (src/inversion/admm.rs:117-119, src/utils/mod.rs:69-77), from the per-block
// FP64 sums (sum d^2, sum x^2) that the TV C2R pass left in V.partial.  One
// block, fixed summation order: repeated runs give identical results.
__device__ __forceinline__ void tv_reduce_block(const VolDesc& V, int gv, VolStatus* status_rw,
                                                VolStatus* mirror, double* sh) {
    typedef double d2v __attribute__((ext_vector_type(2)));
    const QSM_GLOBAL d2v* part = (const QSM_GLOBAL d2v*)glb(V.partial);
    double a = 0.0, b = 0.0;
#pragma unroll 4
    for (int q = threadIdx.x; q < V.npartial; q += kThreads) {
        const d2v v = part[q];
        a += v.x;
        b += v.y;
    }
    const double ta = block_sum(a, sh);
    const double tb = block_sum(b, sh);
    if (threadIdx.x == 0) {
        const double rel = sqrt(ta) / (sqrt(tb) + 1e-20);
        VolStatus st = status_rw[gv];
        st.iters += 1;
        st.rel = rel;
        if (rel < V.tol) st.done = 1;
        status_rw[gv] = st;
        if (mirror) {
            // host-visible copy, read by the host loop after an event wait
            mirror[gv] = st;
            __threadfence_system();
        }
    }
}

__device__ __forceinline__ double fftfreq_at(int i, int n, double d) {
    // src/fft.rs:544-566: index i of numpy fftfreq(n, d)
    const double val = 1.0 / ((double)n * d);
    const int s = (i < (n + 1) / 2) ? i : i - n;
    return (double)s * val;
}

__device__ __forceinline__ int mirror_idx(int i, int n) { return i == 0 ? 0 : n - i; }

// ------------------------------------------------ packed half spectrum --
// A half spectrum stores nxh = (nx + 1) / 2 columns kx.  For even nx the x
// transform of a real row has two real bins, DC and Nyquist (kx = nx/2); both
// go to column 0 as (DC, Nyquist), so every row holds nx/2 complex values and
// the y / z passes work on whole 16-column tiles with rows of nx/2 * 8 bytes.
// Column 0 then carries the kx = 0 plane P0 and the kx = nx/2 plane PN, both
// real in (y, z) and so Hermitian in (ky, kz).  The forward y pass
// separates them: after it, entry ky of column 0 holds
//   ky = 0, ny/2 : P0(ky) + i PN(ky)            (both real in ky, left packed)
//   0 < ky < ny/2: P0(ky)
//   ny/2 < ky    : PN(ny - ky)
// so the z pass sees column 0 at ky < ny/2 as frequency (0, ky), at
// ky > ny/2 as (nx/2, ny - ky), and at ky = 0, ny/2 a column Z = A + i B of
// two z spectra A (kx = 0) and B (kx = nx/2), each Hermitian in kz, which a
// real per-frequency multiplier pair (mA, mB) maps to
//   alpha Z(kz) + beta conj(Z(-kz)),  alpha = (mA + mB)/2, beta = (mA - mB)/2.
// The inverse y pass packs the entries back before transforming.  Odd nx has
// no Nyquist bin and no packing.
__device__ __forceinline__ bool packed_x(const VolDesc& V) { return (V.nx & 1) == 0; }

// Frequency (fx, fy) of column kx of a z-pass tile at ky (not for the two
// doubly packed columns, see pk_double).
__device__ __forceinline__ void pk_freq(const VolDesc& V, int kx, int ky, int& fx, int& fy) {
    const bool nyq = kx == 0 && packed_x(V) && 2 * ky > V.ny;
    fx = nyq ? V.nx / 2 : kx;
    fy = nyq ? V.ny - ky : ky;
}

// Tile tx at ky holds a doubly packed column 0 (block-uniform).
__device__ __forceinline__ bool pk_double(const VolDesc& V, int tx, int ky) {
    return tx == 0 && packed_x(V) && (ky == 0 || 2 * ky == V.ny);
}

// alpha z + beta conj(zm) for the multiplier pair (mA, mB)
__device__ __forceinline__ float2 pk_apply(float2 z, float2 zm, float mA, float mB) {
    const float a = 0.5f * (mA + mB), b = 0.5f * (mA - mB);
    return make_float2(a * z.x + b * zm.x, a * z.y - b * zm.y);
}
__device__ __forceinline__ float2 pk_apply_d(float2 z, float2 zm, double mA, double mB) {
    const double a = 0.5 * (mA + mB), b = 0.5 * (mA - mB);
    return make_float2((float)(a * (double)z.x + b * (double)zm.x), (float)(a * (double)z.y - b * (double)zm.y));
}

// Entry s of column 0 after the forward y transform (w = W(s), wm = W(ny-s)).
__device__ __forceinline__ float2 ypk_fwd(int s, int ny, float2 w, float2 wm) {
    if (s == 0 || 2 * s == ny) return w;
    if (2 * s < ny) return make_float2(0.5f * (w.x + wm.x), 0.5f * (w.y - wm.y));  // P0(s)
    return make_float2(0.5f * (wm.y + w.y), 0.5f * (w.x - wm.x));                  // PN(ny-s)
}
// W(s) rebuilt before the inverse y transform from entries s and ny - s.
__device__ __forceinline__ float2 ypk_inv(int s, int ny, float2 own, float2 mir) {
    if (s == 0 || 2 * s == ny) return own;
    if (2 * s < ny) return make_float2(own.x - mir.y, own.y + mir.x);  // P0(s) + i PN(s)
    return make_float2(mir.x + own.y, own.x - mir.y);                  // conj P0 + i conj PN
}

// The same on column 0 of a tile of TW columns held in LDS (lds[row * TW +
// c], ny <= kMaxLen); every thread of the block calls it.
template <bool INV, int TW = kTile>
__device__ __forceinline__ void ypk_lds(float2* lds, int ny) {
    constexpr int Q = (TW == kTile ? kWideTileMaxLen : kMaxLen) / kThreads;
    float2 own[Q], mir[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int s = min((int)threadIdx.x + q * kThreads, ny - 1);
        own[q] = lds[s * TW];
        mir[q] = lds[mirror_idx(s, ny) * TW];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int s = threadIdx.x + q * kThreads;
        if (s < ny) lds[s * TW] = INV ? ypk_inv(s, ny, own[q], mir[q]) : ypk_fwd(s, ny, own[q], mir[q]);
    }
    __syncthreads();
}

// Binary sphere of src/kernels/smv.rs:19-67 (un-normalised: 1 inside).  The
// squared distance is formed in FP64 in the reference's order with every
// product and sum rounded (contraction off), so boundary voxels are
// classified exactly as the reference (and the host voxel count) do.
__device__ __forceinline__ float sphere_element(const VolDesc& V, int i, int r, int ridx) {
    // The reference rounds every product and sum (no fused multiply-add);
    // with FMA contraction voxels at exactly the radius (e.g. (4,3,0) *
    // 0.9 mm at 4.5 mm) fall outside.  The pragma covers only operations
    // written in this scope (the __dmul_rn / __dadd_rn helpers are still
    // contracted after inlining), so the arithmetic is spelled out here.
#pragma clang fp contract(off)
    const int k = (int)fastdiv((uint32_t)r, V.m_ny);
    const int j = r - k * V.ny;
    const double xi = (i <= V.nx / 2) ? (double)i : (double)(i - V.nx);
    const double yj = (j <= V.ny / 2) ? (double)j : (double)(j - V.ny);
    const double zk = (k <= V.nz / 2) ? (double)k : (double)(k - V.nz);
    const double dx = xi * V.vsx, dy = yj * V.vsy, dz = zk * V.vsz;
    const double dxx = dx * dx, dyy = dy * dy, dzz = dz * dz;
    const double d2 = (dxx + dyy) + dzz;
    const double rad = V.vs_radii[ridx];
    return (d2 <= rad * rad) ? 1.0f : 0.0f;
}

// ---------------------------------------------------------- tile helpers --
// Column tile: element (row, c) at lds[row*TW + c] <-> base[kx0 + c + row*stride];
// columns kx >= nxh read as zero and are not written.
template <int EMAX, int TW = kTile>
__device__ __forceinline__ void col_load(float2* lds, const QSM_GLOBAL float2* __restrict__ base,
                                         size_t stride, int n, int kx0, int nxh) {
    constexpr int L2 = tile_log2(TW);
    float2 r[EMAX];
    const int total = n * TW;
    // unconditional loads: rows past n and columns past nxh read in-bounds
    // elements that are never stored
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        const int row = min(e >> L2, n - 1);
        const int kx = min(kx0 + (e & (TW - 1)), nxh - 1);
        r[t] = ldg2(base + kx + row * stride);
    }
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < total) lds[e] = r[t];
    }
}

template <int EMAX, int TW = kTile>
__device__ __forceinline__ void col_store(const float2* lds, QSM_GLOBAL float2* __restrict__ base,
                                          size_t stride, int n, int kx0, int nxh) {
    constexpr int L2 = tile_log2(TW);
    const int total = n * TW;
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        const int row = e >> L2;
        const int kx = kx0 + (e & (TW - 1));
        if (e < total && kx < nxh) stg2(base + kx + row * stride, lds[e]);
    }
}

// Tile I/O in the register layouts of fft_col2.hpp (thread (j, c) = (t >> 4,
// t & 15), column kx0 + c).  L16: rows j + 16 r, r < R0; LR: rows j + R0 r,
// r < 16, threads j < R0.  Columns kx >= nxh load column nxh - 1 (in bounds,
// their results are never stored) and are not written.
static_assert(kTile == 16 && kThreads == 256, "fft_col2.hpp assumes 16-column tiles and 256 threads");

// The TV / RTS z-pass operands f^ (SPEC_A) and q are written once at setup
// and read at every iteration by the same z-pass block, so they are stored
// tile-major: the tile of TW columns at (tx, ky) holds its nz rows of TW
// elements contiguously.  Element (kx, kz) of that tile is at
// zop_base(...) + kx + kz * TW.
__host__ __device__ inline size_t zop_base(int ky, int tx, int ntx, int nz, int TW) {
    return ((size_t)ky * ntx + tx) * (size_t)nz * TW - (size_t)tx * TW;
}

template <int R0>
__device__ __forceinline__ void l16_load(float2 (&v)[16], const QSM_GLOBAL float2* __restrict__ base,
                                         size_t stride, int kx0, int nxh) {
    const int c = threadIdx.x & 15, j = threadIdx.x >> 4;
    const int kx = min(kx0 + c, nxh - 1);
    const QSM_GLOBAL float2* p = base + kx + (size_t)j * stride;
#pragma unroll
    for (int r = 0; r < R0; ++r) v[r] = ldg2(p + (size_t)(16 * r) * stride);
}

template <int R0>
__device__ __forceinline__ void l16_store(const float2 (&v)[16], QSM_GLOBAL float2* __restrict__ base,
                                          size_t stride, int kx0, int nxh) {
    const int c = threadIdx.x & 15, j = threadIdx.x >> 4;
    const int kx = kx0 + c;
    if (kx >= nxh) return;
    QSM_GLOBAL float2* p = base + kx + (size_t)j * stride;
#pragma unroll
    for (int r = 0; r < R0; ++r) stg2(p + (size_t)(16 * r) * stride, v[r]);
}

template <int R0>
__device__ __forceinline__ void lr_store(const float2 (&v)[16], QSM_GLOBAL float2* __restrict__ base,
                                         size_t stride, int kx0, int nxh) {
    const int c = threadIdx.x & 15, j = threadIdx.x >> 4;
    const int kx = kx0 + c;
    if (kx >= nxh || j >= R0) return;
    QSM_GLOBAL float2* p = base + kx + (size_t)j * stride;
#pragma unroll
    for (int r = 0; r < 16; ++r) stg2(p + (size_t)(R0 * r) * stride, v[r]);
}

// ------------------------------------------------ x-pass source fills ----
enum SrcKind : int {
    SRC_F64 = 0, SRC_U8 = 1, SRC_F32 = 2, SRC_SPHERE = 3, SRC_TVDIV = 4,
    SRC_TVDIV_REC = 5,    // SRC_TVDIV that also records the shrink pattern
    SRC_TVADJ_FIRST = 6,  // adjoint source of the last iteration: x-bar = mask * chi-bar
    SRC_TVADJ = 7,        // adjoint source of an earlier iteration
    SRC_ACC = 8,          // the adjoint accumulator
    SRC_X0 = 9,           // x[0] (the RTS starting point)
    SRC_WRAPLAP = 10,     // masked wrapped Laplacian of the f64 phase in field
    SRC_TVDIV_W = 11,     // SRC_TVDIV with NLTV weights (buffer ck)
    SRC_NLTV_BND = 12     // first step of a later NLTV Newton round (previous weights ck)
};

// wrap into [-pi, pi] as src/unwrap/laplacian.rs:41-50 (f64 remainder).
__device__ __forceinline__ double wrap_pi(double x) {
    const double two_pi = 6.283185307179586476925286766559;
    const double pi = 3.14159265358979323846264338327950288;
    double y = fmod(x, two_pi);
    if (y > pi) y -= two_pi;
    else if (y < -pi) y += two_pi;
    return y;
}

// Wrapped periodic Laplacian at voxel (i, row r), zero outside the mask
// (src/unwrap/laplacian.rs:67-122 and the masking of :146-150), in FP64.
__device__ __forceinline__ float wraplap_at(const VolDesc& V, int i, int r) {
#pragma clang fp contract(off)
    const int nx = V.nx, ny = V.ny, nz = V.nz;
    const size_t idx = i + (size_t)r * nx;
    if (!glb(V.mask)[idx]) return 0.0f;
    const int k = (int)fastdiv((uint32_t)r, V.m_ny);
    const int j = r - k * ny;
    const size_t nxy = (size_t)nx * ny;
    auto at = [&](int ii, int jj, int kk) { return glb(V.field)[ii + (size_t)jj * nx + (size_t)kk * nxy]; };
    const double u = at(i, j, k);
    const double uxp = at(i + 1 < nx ? i + 1 : 0, j, k), uxm = at(i > 0 ? i - 1 : nx - 1, j, k);
    const double uyp = at(i, j + 1 < ny ? j + 1 : 0, k), uym = at(i, j > 0 ? j - 1 : ny - 1, k);
    const double uzp = at(i, j, k + 1 < nz ? k + 1 : 0), uzm = at(i, j, k > 0 ? k - 1 : nz - 1);
    const double dx2 = 1.0 / (V.vsx * V.vsx), dy2 = 1.0 / (V.vsy * V.vsy), dz2 = 1.0 / (V.vsz * V.vsz);
    const double lx = (wrap_pi(uxp - u) - wrap_pi(u - uxm)) * dx2;
    const double ly = (wrap_pi(uyp - u) - wrap_pi(u - uym)) * dy2;
    const double lz = (wrap_pi(uzp - u) - wrap_pi(u - uzm)) * dz2;
    return (float)(lx + ly + lz);
}

template <int SRC>
__device__ __forceinline__ float simple_src(const VolDesc& V, int i, int r, int aux) {
    if constexpr (SRC == SRC_F64) return (float)glb(V.field)[i + (size_t)r * V.nx];
    else if constexpr (SRC == SRC_U8) return (float)glb(V.mask)[i + (size_t)r * V.nx];
    else if constexpr (SRC == SRC_F32) return glb(V.vs_local)[i + (size_t)r * V.nx];
    else if constexpr (SRC == SRC_ACC) return glb(V.adj_acc)[i + (size_t)r * V.nx];
    else if constexpr (SRC == SRC_X0) return glb(V.x[0])[i + (size_t)r * V.nx];
    else if constexpr (SRC == SRC_WRAPLAP) return wraplap_at(V, i, r);
    else return sphere_element(V, i, r, aux);
}

// lds[p*nx + i] = (row 2p, row 2p+1) of the block's rows.
template <int N, int EMAX, int SRC>
__device__ __forceinline__ void fill_simple(float2* lds, const VolDesc& V, int nx, int RB, int row0,
                                            int nrows, int aux) {
    const int total = RB * nx;
    float2 r[EMAX];
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        const int p = div_nx<N>(e, V);
        const int i = e - p * nx;
        const int ra = row0 + 2 * p, rb = ra + 1;
        r[t].x = (e < total && ra < nrows) ? simple_src<SRC>(V, i, ra, aux) : 0.0f;
        r[t].y = (e < total && rb < nrows) ? simple_src<SRC>(V, i, rb, aux) : 0.0f;
    }
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < total) lds[e] = r[t];
    }
}

// Divergence of g = 2z - v for the z/u update fused in front of the
// x-subproblem: v = grad(x) + u (periodic forward differences,
// src/utils/gradient.rs:21-58), z = shrink(v, lambda/rho), u' = v - z,
// g = 2z - v (src/inversion/admm.rs:127-142), div = bdiv(g)
// (src/utils/gradient.rs:71-108).  The x component of g at i-1 is recomputed
// from x and u at i-1 (likewise y and z), so g never goes to memory.
// CH elements (2*CH voxels) per round, all their loads issued before the
// arithmetic; restrict-qualified so the u' stores of one round do not order
// the next round's loads.
// The operands of CH elements (2*CH voxels) of the divergence.
// W: per-voxel shrink weights (NLTV, weighted_shrink of src/utils/mod.rs:
// 55-59): wv = w at i, i-e_x, i-e_y, i-e_z.
template <int CH, bool W = false>
struct TvDivRound {
    float xv[CH][2][7], uv[CH][2][6];
    float wv[CH][2][W ? 4 : 1];
    int idx[CH][2];
    bool ok[CH][2];
};

template <int CH, bool W = false>
__device__ __forceinline__ void tvdiv_load(TvDivRound<CH, W>& R, const VolDesc& V, int nx, int t0, int EMAX,
                                           int total, int row0, int nrows,
                                           const QSM_GLOBAL float* __restrict__ x,
                                           const QSM_GLOBAL float* __restrict__ u,
                                           const QSM_GLOBAL float* __restrict__ w = nullptr) {
    const int ny = V.ny, nz = V.nz;
    const int nxy = nx * ny, N = nxy * nz;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e = threadIdx.x + (t0 + c) * kThreads;
        const int p = e / nx;
        const int i = e - p * nx;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = row0 + 2 * p + h;
            const bool ok = (t0 + c < EMAX) && (e < total) && (r < nrows);
            R.ok[c][h] = ok;
            const int rr = ok ? r : 0;
            const int ii = ok ? i : 0;
            const int k = (int)fastdiv((uint32_t)rr, V.m_ny);
            const int j = rr - k * ny;
            const int idx = ii + rr * nx;
            R.idx[c][h] = idx;
            const int dxp = (ii + 1 < nx) ? 1 : 1 - nx;
            const int dxm = (ii > 0) ? -1 : nx - 1;
            const int dyp = (j + 1 < ny) ? nx : nx - nxy;
            const int dym = (j > 0) ? -nx : nxy - nx;
            const int dzp = (k + 1 < nz) ? nxy : nxy - N;
            const int dzm = (k > 0) ? -nxy : N - nxy;
            R.xv[c][h][0] = x[idx];
            R.xv[c][h][1] = x[idx + dxp];
            R.xv[c][h][2] = x[idx + dyp];
            R.xv[c][h][3] = x[idx + dzp];
            R.xv[c][h][4] = x[idx + dxm];
            R.xv[c][h][5] = x[idx + dym];
            R.xv[c][h][6] = x[idx + dzm];
            R.uv[c][h][0] = u[idx];
            R.uv[c][h][1] = u[N + idx];
            R.uv[c][h][2] = u[2 * N + idx];
            R.uv[c][h][3] = u[idx + dxm];
            R.uv[c][h][4] = u[N + idx + dym];
            R.uv[c][h][5] = u[2 * N + idx + dzm];
            if constexpr (W) {
                R.wv[c][h][0] = w[idx];
                R.wv[c][h][1] = w[idx + dxm];
                R.wv[c][h][2] = w[idx + dym];
                R.wv[c][h][3] = w[idx + dzm];
            }
        }
    }
}

__device__ __forceinline__ int8_t shrink_sign(float v, float t) {
    return v > t ? (int8_t)1 : (v < -t ? (int8_t)-1 : (int8_t)0);
}

template <int CH, bool REC, bool W, bool NT>
__device__ __forceinline__ void tvdiv_compute(const TvDivRound<CH, W>& R, float2* lds, const VolDesc& V,
                                              int t0, int EMAX, int total,
                                              QSM_GLOBAL float* __restrict__ uo,
                                              QSM_GLOBAL int8_t* __restrict__ rec, float wnorm = 1.0f) {
    const int N = V.nx * V.ny * V.nz;
    const float t = V.thr, hx = V.hx, hy = V.hy, hz = V.hz;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e = threadIdx.x + (t0 + c) * kThreads;
        float d[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float xc = R.xv[c][h][0];
            const float vx = (R.xv[c][h][1] - xc) * hx + R.uv[c][h][0];
            const float vy = (R.xv[c][h][2] - xc) * hy + R.uv[c][h][1];
            const float vz = (R.xv[c][h][3] - xc) * hz + R.uv[c][h][2];
            const float vxm = (xc - R.xv[c][h][4]) * hx + R.uv[c][h][3];
            const float vym = (xc - R.xv[c][h][5]) * hy + R.uv[c][h][4];
            const float vzm = (xc - R.xv[c][h][6]) * hz + R.uv[c][h][5];
            // thresholds lambda/rho, times the weight (divided by its
            // normalisation) of the voxel each component belongs to
            float ti = t, txm = t, tym = t, tzm = t;
            if constexpr (W) {
                ti = t * (R.wv[c][h][0] / wnorm);
                txm = t * (R.wv[c][h][1] / wnorm);
                tym = t * (R.wv[c][h][2] / wnorm);
                tzm = t * (R.wv[c][h][3] / wnorm);
            }
            const float zx = shrinkf(vx, ti), zy = shrinkf(vy, ti), zz = shrinkf(vz, ti);
            if (R.ok[c][h]) {
                const int idx = R.idx[c][h];
                stx<NT>(uo + idx, vx - zx);
                stx<NT>(uo + N + idx, vy - zy);
                stx<NT>(uo + 2 * N + idx, vz - zz);
                if constexpr (REC) {
                    // d z / d v of this update, for the unrolled adjoint
                    rec[idx] = shrink_sign(vx, t);
                    rec[N + idx] = shrink_sign(vy, t);
                    rec[2 * N + idx] = shrink_sign(vz, t);
                }
            }
            const float gx = 2.0f * zx - vx, gy = 2.0f * zy - vy, gz = 2.0f * zz - vz;
            const float gxm = 2.0f * shrinkf(vxm, txm) - vxm;
            const float gym = 2.0f * shrinkf(vym, tym) - vym;
            const float gzm = 2.0f * shrinkf(vzm, tzm) - vzm;
            d[h] = R.ok[c][h] ? (gx - gxm) * hx + (gy - gym) * hy + (gz - gzm) * hz : 0.0f;
        }
        if (t0 + c < EMAX && e < total) lds[e] = make_float2(d[0], d[1]);
    }
}

// Divergence of g = 2z - v for the z/u update fused in front of the
// x-subproblem: v = grad(x) + u (periodic forward differences,
// src/utils/gradient.rs:21-58), z = shrink(v, lambda/rho), u' = v - z,
// g = 2z - v (src/inversion/admm.rs:127-142), div = bdiv(g)
// (src/utils/gradient.rs:71-108).  The x component of g at i-1 is recomputed
// from x and u at i-1 (likewise y and z), so g never goes to memory.
// Rounds of CH elements (2*CH voxels) are software-pipelined: the loads of
// round r+1 are issued before round r is computed and stored.
// RT: row length and rows known at run time only.  Such a block may fill a small
// part of its tile, so the fills end with its elements: each round past them had
// every thread load voxel 0 and its neighbours (six volumes of 16x64x48, 10
// unrolled iterations and their gradient in blocks of 8 rows: 1.06 ms with those
// rounds, 0.85 without).
template <int EMAX, bool REC, bool W, bool NT, bool RT>
__device__ __forceinline__ void fill_tvdiv(float2* lds, const VolDesc& V, int nx, int RB,
                                           const QSM_GLOBAL float* __restrict__ x,
                                           const QSM_GLOBAL float* __restrict__ u,
                                           QSM_GLOBAL float* __restrict__ uo, int row0, int nrows,
                                           QSM_GLOBAL int8_t* __restrict__ rec,
                                           const QSM_GLOBAL float* __restrict__ w = nullptr,
                                           float wnorm = 1.0f) {
    constexpr int CH = (W || EMAX <= kRowEmaxRt) ? 1 : 2;
    constexpr int NR = (EMAX + CH - 1) / CH;
    const int total = RB * nx;
    // round r holds elements of the block (a constant where N is)
    auto has = [&](int r) { return r < NR && (!RT || r * CH * kThreads < total); };
    TvDivRound<CH, W> A, B;
    tvdiv_load<CH, W>(A, V, nx, 0, EMAX, total, row0, nrows, x, u, w);
#pragma unroll
    for (int r = 0; r < NR; r += 2) {
        if (RT && !has(r)) break;
        if (has(r + 1)) tvdiv_load<CH, W>(B, V, nx, (r + 1) * CH, EMAX, total, row0, nrows, x, u, w);
        tvdiv_compute<CH, REC, W, NT>(A, lds, V, r * CH, EMAX, total, uo, rec, wnorm);
        if (has(r + 1)) {
            if (has(r + 2)) tvdiv_load<CH, W>(A, V, nx, (r + 2) * CH, EMAX, total, row0, nrows, x, u, w);
            tvdiv_compute<CH, REC, W, NT>(B, lds, V, (r + 1) * CH, EMAX, total, uo, rec, wnorm);
        }
    }
}

// Lane rotations across the 64-wide wavefront (DPP wave_rol / wave_ror):
// lane l receives the value of lane l + 1 (lane_next) or l - 1 (lane_prev),
// modulo 64.
__device__ __forceinline__ float lane_next(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x134, 0xF, 0xF,
                                                                 false));
}
__device__ __forceinline__ float lane_prev(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x13C, 0xF, 0xF,
                                                                 false));
}

// Row lengths and pair-rows per block (RB) the wave-row form takes: at
// least one pair-row per wave, at most 4 column groups per lane.  Measured
// (one column per lane): faster than the element-wise fill at 144 ... 256;
// at 384 (6 groups of 64, 222 VGPRs) slower, and with 7 or 8 groups its two
// row buffers take all 256 VGPRs (one wave per SIMD, where the element-wise
// fill keeps two).  With two columns per lane, 384 takes 178 VGPRs (2 waves
// per SIMD against the element-wise fill's 3) and its TV-ADMM ran 9.0 ->
// 8.8 solves/s; 512 takes 234.
__host__ __device__ constexpr bool tvdiv_rows_form(int n, int rb) {
    return n > 0 && n <= 256 && rb >= 4;
}

// Columns per lane of the wave-row form (VW): 4 above 128 columns and 2 from 66
// to 128, one group of lanes for the row, so that every load and store moves 16
// or 8 bytes per lane; 1 for other rows.  Measured at 256, one column per lane
// against 2 and 4: 277.9, 274.8 and 268.2 us per 4-volume launch; at 144 (three
// groups of 64 columns against 36 lanes of 4) 78.8 and 71.6 us for two
// 144x192x160 volumes, at 160 81.4 and 79.0, at 176 91.7 and 88.1, at 192 the
// same.  Two groups of 2 lose to three of 1 (150 columns: 142 registers against
// 117, 23.2 us against 19.8 at 150x144x96).
__host__ __device__ constexpr int tvdiv_rows_vw(int n) {
    return n % 4 == 0 && n > 128 ? 4 : (n % 2 == 0 && n > 64 && n <= 128 ? 2 : 1);
}

template <int VW>
using lanev = std::conditional_t<VW == 1, float, std::conditional_t<VW == 2, float2, float4>>;
typedef float qsm_f4v __attribute__((ext_vector_type(4)));
// element e (a compile-time constant after unrolling) of a lane's columns
template <int VW>
__device__ __forceinline__ float vel(const lanev<VW>& v, int e) {
    if constexpr (VW == 1) return v;
    else if constexpr (VW == 2) return e == 0 ? v.x : v.y;
    else return e == 0 ? v.x : (e == 1 ? v.y : (e == 2 ? v.z : v.w));
}
template <int VW>
__device__ __forceinline__ lanev<VW> vpack(const float (&a)[VW]) {
    if constexpr (VW == 1) return a[0];
    else if constexpr (VW == 2) return make_float2(a[0], a[1]);
    else return make_float4(a[0], a[1], a[2], a[3]);
}
template <int VW>
__device__ __forceinline__ float vfirst(const lanev<VW>& v) { return vel<VW>(v, 0); }
template <int VW>
__device__ __forceinline__ float vlast(const lanev<VW>& v) { return vel<VW>(v, VW - 1); }
template <int VW>
__device__ __forceinline__ lanev<VW> vzero() {
    const float z[VW] = {};
    return vpack<VW>(z);
}
template <int VW, bool NT = false>
__device__ __forceinline__ lanev<VW> ldv(const QSM_GLOBAL float* p) {
    if constexpr (VW == 1) return ldx<NT>(p);
    else if constexpr (VW == 2) return ldg2<NT>((const QSM_GLOBAL float2*)p);
    else {
        const qsm_f4v v = ldx<NT>((const QSM_GLOBAL qsm_f4v*)p);
        return make_float4(v.x, v.y, v.z, v.w);
    }
}
template <int VW, bool NT = false>
__device__ __forceinline__ void stv(QSM_GLOBAL float* p, lanev<VW> v) {
    if constexpr (VW == 1) {
        stx<NT>(p, v);
    } else if constexpr (VW == 2) {
        qsm_f2v w;
        w.x = v.x;
        w.y = v.y;
        stx<NT>((QSM_GLOBAL qsm_f2v*)p, w);
    } else {
        qsm_f4v w;
        w.x = v.x;
        w.y = v.y;
        w.z = v.z;
        w.w = v.w;
        stx<NT>((QSM_GLOBAL qsm_f4v*)p, w);
    }
}

// One row of the wave-row form below: lane l holds columns VW l ... VW l +
// VW - 1 of each group of G = 64 VW columns, m < C = ceil(NX / G) (in a
// partial last group the lanes past the row's end hold its last VW columns
// again and are never stored).
template <int NX, int VW>
struct TvRow {
    static constexpr int G = 64 * VW;
    static constexpr int C = (NX + G - 1) / G;
    lanev<VW> xc[C], ux[C], uy[C], uz[C], xzp[C], xzm[C], uzm[C];
};

// first column of the lane's set in group m
template <int NX, int VW>
__device__ __forceinline__ int tv_col(int lane, int m) {
    constexpr int G = 64 * VW, C = (NX + G - 1) / G;
    return (NX % G != 0 && m == C - 1) ? min(VW * lane + G * m, NX - VW) : VW * lane + G * m;
}

// Row r of the volume (r = j + k ny, k the plane): its own x and u, x on the
// planes k +- 1 and u_z on plane k - 1 (periodic).
template <int NX, int VW, bool NT>
__device__ __forceinline__ void tvrow_load(TvRow<NX, VW>& R, int r, int k, int nz, int nxy, int N, int lane,
                                           const QSM_GLOBAL float* __restrict__ x,
                                           const QSM_GLOBAL float* __restrict__ u) {
    constexpr int C = TvRow<NX, VW>::C;
    const int base = r * NX;
    const int dzp = (k + 1 < nz) ? nxy : nxy - N;
    const int dzm = (k > 0) ? -nxy : N - nxy;
    const QSM_GLOBAL float* xr = x + base;
    const QSM_GLOBAL float* ur = u + base;
#pragma unroll
    for (int m = 0; m < C; ++m) R.xc[m] = ldv<VW>(xr + tv_col<NX, VW>(lane, m));
#pragma unroll
    for (int m = 0; m < C; ++m) {
        const int i = tv_col<NX, VW>(lane, m);
        R.ux[m] = ldv<VW, NT>(ur + i);
        R.uy[m] = ldv<VW, NT>(ur + N + i);
        R.uz[m] = ldv<VW>(ur + 2 * N + i);
        R.xzp[m] = ldv<VW>(xr + dzp + i);
        R.xzm[m] = ldv<VW>(xr + dzm + i);
        R.uzm[m] = ldv<VW>(ur + 2 * N + dzm + i);
    }
}

// One component of the z/u update for a threshold t >= 0: with z =
// shrink(v, t), u' = v - z is v clamped to [-t, t] (one v_med3) and g = 2z - v
// = v - 2u'.  tvdiv_compute's form (two compares and selects, then v - z and
// 2z - v) took 7 instructions more per component, six components a voxel,
// and VALU issue was a third of the pass's time.
__device__ __forceinline__ float tv_clamp(float v, float t) { return __builtin_amdgcn_fmed3f(v, -t, t); }
__device__ __forceinline__ float tv_g(float v, float u) { return fmaf(-2.0f, u, v); }
__device__ __forceinline__ float tv_gv(float v, float t) { return tv_g(v, tv_clamp(v, t)); }

// fill_tvdiv (t >= 0) with the block's RB pair-rows split over its four
// waves: wave w takes pair-rows [w RB / 4, (w + 1) RB / 4), lane l the columns
// VW l ... VW l + VW - 1 (+ 64 VW m).  Row indices are then the same in every
// lane (scalar).  x right of the lane's last column comes from a lane rotation
// (lane l + 1); g's x component left of its first column from lane l - 1, and
// its y component one row up from the wave's previous row, both already
// formed (with a partial last column group, the periodic wrap between columns
// NX - 1 and 0 from lane broadcasts); only the rows above and below the wave's
// rows, and y-wrapping rows, are loaded again.  Loads per voxel: 7 plus 3 /
// (rows per wave), against 13.
template <int NX, int RB, bool NT>
__device__ __forceinline__ void fill_tvdiv_rows(float2* lds, const VolDesc& V, int row0, int nrows,
                                                const QSM_GLOBAL float* __restrict__ x,
                                                const QSM_GLOBAL float* __restrict__ u,
                                                QSM_GLOBAL float* __restrict__ uo) {
    constexpr int VW = tvdiv_rows_vw(NX);
    using vt = lanev<VW>;
    constexpr int G = TvRow<NX, VW>::G;
    constexpr int C = TvRow<NX, VW>::C;
    constexpr int LV = (NX - G * (C - 1)) / VW;  // valid lanes of the last column group
    static_assert(kThreads == 256, "four waves per block");
    static_assert(VW == 1 || C == 1, "several columns per lane: one group of lanes");
    const int ny = V.ny, nz = V.nz;
    const int nxy = NX * ny, N = nxy * nz;
    const float t = V.thr, hx = V.hx, hy = V.hy, hz = V.hz;
    const int lane = (int)(threadIdx.x & 63);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // pair-rows [p0, p0 + nrw / 2) of this wave
    static_assert(RB % 4 == 0, "the same rows for every wave");
    const int p0 = wv * (RB / 4);
    constexpr int nrw = RB / 2;
    const int r0 = row0 + 2 * p0;
    // plane and in-plane index of the wave's first row, then stepped
    int k = r0 / ny;
    int j = r0 - k * ny;
    TvRow<NX, VW> A, B;
    vt hym_x[C], hym_uy[C], hyp_x[C];  // rows above / below the wave's rows
    if (r0 < nrows) {
        tvrow_load<NX, VW, NT>(A, r0, k, nz, nxy, N, lane, x, u);
        // the row before the wave's first row, periodic in y
        const int ra = j > 0 ? r0 - 1 : r0 + ny - 1;
        const QSM_GLOBAL float* xr = x + ra * NX;
        const QSM_GLOBAL float* ur = u + N + ra * NX;
#pragma unroll
        for (int m = 0; m < C; ++m) {
            hym_x[m] = ldv<VW>(xr + tv_col<NX, VW>(lane, m));
            hym_uy[m] = ldv<VW>(ur + tv_col<NX, VW>(lane, m));
        }
    } else {
#pragma unroll
        for (int m = 0; m < C; ++m) hym_x[m] = hym_uy[m] = vzero<VW>();
    }
    vt pgy[C], dev[C];  // g's y component in the previous row; the pair's first row
    // row q of the wave from cur, with the next row's loads issued into nxt;
    // ODD: the second row of a pair-row (the pair goes to LDS)
    auto step = [&](TvRow<NX, VW>& cur, TvRow<NX, VW>& nxt, const int q, auto odd) {
        constexpr bool ODD = decltype(odd)::value;
        const int r = r0 + q;
        const bool ok = r < nrows;
        // plane / in-plane index of row r + 1
        int jn = j + 1, kn = k;
        if (jn == ny) {
            jn = 0;
            ++kn;
        }
        if (q + 1 < nrw && r + 1 < nrows) tvrow_load<NX, VW, NT>(nxt, r + 1, kn, nz, nxy, N, lane, x, u);
        if (q + 2 == nrw && ok) {
            // the row after the wave's last row rl = r + 1 (in-plane index
            // jn), periodic in y; issued one row ahead
            const int rl = r + 1;
            const bool okl = rl < nrows;
            const int rb = (jn + 1 < ny) ? rl + 1 : rl - ny + 1;
            const QSM_GLOBAL float* xr = x + (okl ? rb : 0) * NX;
#pragma unroll
            for (int m = 0; m < C; ++m) hyp_x[m] = okl ? ldv<VW>(xr + tv_col<NX, VW>(lane, m)) : vzero<VW>();
        }
        vt gym[C], xyp[C];
        // g's y component at y - 1 where it is not the wave's previous row
        auto gy_at = [&](const vt& xc, const vt& xm, const vt& um) {
            float g[VW];
#pragma unroll
            for (int e = 0; e < VW; ++e) g[e] = tv_gv((vel<VW>(xc, e) - vel<VW>(xm, e)) * hy + vel<VW>(um, e), t);
            return vpack<VW>(g);
        };
        if (!ok) {
            // rows past the volume (the last block): d = 0, nothing stored
#pragma unroll
            for (int m = 0; m < C; ++m) {
                gym[m] = xyp[m] = vzero<VW>();
                cur.xc[m] = cur.ux[m] = cur.uy[m] = cur.uz[m] = vzero<VW>();
                cur.xzp[m] = cur.xzm[m] = cur.uzm[m] = vzero<VW>();
            }
        } else {
            // y - 1
            if (q == 0) {
#pragma unroll
                for (int m = 0; m < C; ++m) gym[m] = gy_at(cur.xc[m], hym_x[m], hym_uy[m]);
            } else if (j == 0) {
                const int ra = r + ny - 1;
#pragma unroll
                for (int m = 0; m < C; ++m)
                    gym[m] = gy_at(cur.xc[m], ldv<VW>(x + ra * NX + tv_col<NX, VW>(lane, m)),
                                   ldv<VW>(u + N + ra * NX + tv_col<NX, VW>(lane, m)));
            } else {
#pragma unroll
                for (int m = 0; m < C; ++m) gym[m] = pgy[m];
            }
            // y + 1
            if (q + 1 == nrw) {
#pragma unroll
                for (int m = 0; m < C; ++m) xyp[m] = hyp_x[m];
            } else if (j + 1 == ny) {
                const int rb = r - ny + 1;
#pragma unroll
                for (int m = 0; m < C; ++m) xyp[m] = ldv<VW>(x + rb * NX + tv_col<NX, VW>(lane, m));
            } else {
#pragma unroll
                for (int m = 0; m < C; ++m) xyp[m] = nxt.xc[m];
            }
        }
        // x right of the lane's last column from lane l + 1 (lane 63: lane 0
        // of the next column group); column NX - 1's right neighbour is
        // column 0 (whole groups: the rotation wraps by itself; a partial
        // last group: from a lane broadcast)
        float rn[C];
#pragma unroll
        for (int m = 0; m < C; ++m) rn[m] = lane_next(vfirst<VW>(cur.xc[m]));
        [[maybe_unused]] float x0 = 0.0f;
        if constexpr (NX % G != 0)
            x0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, vfirst<VW>(cur.xc[0])), 0));
        // the x component of every column of the row, then its left neighbour
        // (lane l - 1; lane 0: lane 63 of the previous group)
        float gx[C][VW], ox[C][VW], gl[C];
#pragma unroll
        for (int m = 0; m < C; ++m) {
            float xp = lane == 63 ? rn[(m + 1) % C] : rn[m];
            if constexpr (NX % G != 0) {
                if (m == C - 1 && lane == LV - 1) xp = x0;
            }
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const float xr = e + 1 < VW ? vel<VW>(cur.xc[m], e + 1) : xp;
                const float vx = (xr - vel<VW>(cur.xc[m], e)) * hx + vel<VW>(cur.ux[m], e);
                ox[m][e] = tv_clamp(vx, t);
                gx[m][e] = tv_g(vx, ox[m][e]);
            }
        }
#pragma unroll
        for (int m = 0; m < C; ++m) gl[m] = lane_prev(gx[m][VW - 1]);
        [[maybe_unused]] float glast = 0.0f;
        if constexpr (NX % G != 0)
            glast = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gx[C - 1][VW - 1]), LV - 1));
        vt d[C];
#pragma unroll
        for (int m = 0; m < C; ++m) {
            float gxm0 = lane == 0 ? gl[(m + C - 1) % C] : gl[m];
            if constexpr (NX % G != 0) {
                if (m == 0 && lane == 0) gxm0 = glast;
            }
            const bool col_ok = NX % G == 0 || m < C - 1 || lane < LV;
            QSM_GLOBAL float* o = uo + r * NX + VW * lane + G * m;
            float oy[VW], oz[VW], gyv[VW], dd[VW];
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const float xc = vel<VW>(cur.xc[m], e);
                const float vy = (vel<VW>(xyp[m], e) - xc) * hy + vel<VW>(cur.uy[m], e);
                const float vz = (vel<VW>(cur.xzp[m], e) - xc) * hz + vel<VW>(cur.uz[m], e);
                const float vzm = (xc - vel<VW>(cur.xzm[m], e)) * hz + vel<VW>(cur.uzm[m], e);
                oy[e] = tv_clamp(vy, t);
                oz[e] = tv_clamp(vz, t);
                gyv[e] = tv_g(vy, oy[e]);
                const float gz = tv_g(vz, oz[e]), gzm = tv_gv(vzm, t);
                const float gxm = e > 0 ? gx[m][e - 1] : gxm0;
                dd[e] = (gx[m][e] - gxm) * hx + (gyv[e] - vel<VW>(gym[m], e)) * hy + (gz - gzm) * hz;
            }
            if (ok && col_ok) {
                stv<VW, NT>(o, vpack<VW>(ox[m]));
                stv<VW, NT>(o + N, vpack<VW>(oy));
                stv<VW, NT>(o + 2 * N, vpack<VW>(oz));
            }
            pgy[m] = vpack<VW>(gyv);
            d[m] = ok ? vpack<VW>(dd) : vzero<VW>();
        }
        if constexpr (ODD) {
            const int p = p0 + (q >> 1);
#pragma unroll
            for (int m = 0; m < C; ++m) {
                const bool col_ok = NX % G == 0 || m < C - 1 || lane < LV;
                if (col_ok) {
                    float2* l2 = lds + p * NX + VW * lane + G * m;
#pragma unroll
                    for (int e = 0; e < VW; ++e) l2[e] = make_float2(vel<VW>(dev[m], e), vel<VW>(d[m], e));
                }
            }
        } else {
#pragma unroll
            for (int m = 0; m < C; ++m) dev[m] = d[m];
        }
        j = jn;
        k = kn;
    };
    // pair-rows of this wave (nrw / 2, wave-uniform): the row
    // buffers keep fixed roles, so nothing is indexed at run time
#pragma unroll
    for (int s = 0; s < (nrw >> 1); ++s) {
        step(A, B, 2 * s, std::false_type{});
        step(B, A, 2 * s + 1, std::true_type{});
    }
}

// VW floats at a 4-byte aligned address (one load / store; global memory
// takes dword alignment).
template <int VW>
struct alignas(4) FloatsU {
    float v[VW];
};
template <int VW, bool NT = false>
__device__ __forceinline__ FloatsU<VW> ldu(const QSM_GLOBAL float* p) {
    if constexpr (VW == 1) {
        return FloatsU<VW>{{ldx<NT>(p)}};
    } else {
        typedef float vt __attribute__((ext_vector_type(VW), aligned(4)));
        const vt w = ldx<NT>((const QSM_GLOBAL vt*)p);
        FloatsU<VW> r;
#pragma unroll
        for (int e = 0; e < VW; ++e) r.v[e] = w[e];
        return r;
    }
}
template <int VW, bool NT>
__device__ __forceinline__ void stu(QSM_GLOBAL float* p, const float (&a)[VW]) {
    if constexpr (VW == 1) {
        stx<NT>(p, a[0]);
    } else {
        typedef float vt __attribute__((ext_vector_type(VW), aligned(4)));
        vt w;
#pragma unroll
        for (int e = 0; e < VW; ++e) w[e] = a[e];
        stx<NT>((QSM_GLOBAL vt*)p, w);
    }
}

// The operands of one row of fill_tvdiv_any in a lane's VW columns, and x and
// u_x at the row's ends (x0, xl, ul: columns 0 and nx - 1), every lane the same.
template <int VW>
struct TvAnyRow {
    FloatsU<VW> xc, ux, uy, uz, xzp, xzm, uzm;
    float x0, xl, ul;
};

// fill_tvdiv (t >= 0) for row lengths known only at run time, in the manner of
// fill_tvdiv_rows: wave w takes the rows [w nr / 4, (w + 1) nr / 4) of the
// block's nr = 2 RB, lane l VW consecutive columns.  Rows up to 64 VW columns
// are one group; longer ones run group by group, 63 VW columns in the first
// (its last lane only lends its x to the right) and 62 VW in each further one
// (lane 0 lends g's x component besides).  A lane's columns past the row's end
// are the next row's first ones: loaded (the buffers end in kRowSlack floats),
// never used.  The periodic neighbours of columns 0 and nx - 1 come from the
// row's end values.  Rows need not be aligned.
// One column per lane with the in-row neighbours loaded took 300 instructions
// per row of 164 columns and 84 us of a pass whose bytes take 36 us.
template <int VW, bool NT>
__device__ __forceinline__ void fill_tvdiv_any(float2* lds, const VolDesc& V, int nx, int RB, int row0,
                                               int nrows, const QSM_GLOBAL float* __restrict__ x,
                                               const QSM_GLOBAL float* __restrict__ u,
                                               QSM_GLOBAL float* __restrict__ uo) {
    using Row = TvAnyRow<VW>;
    const int ny = V.ny, nz = V.nz;
    const int nxy = nx * ny, N = nxy * nz;
    const float t = V.thr, hx = V.hx, hy = V.hy, hz = V.hz;
    const int lane = (int)(threadIdx.x & 63);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int q0 = (wv * 2 * RB) >> 2, q1 = ((wv + 1) * 2 * RB) >> 2;
    const int qe = min(q1, nrows - row0);  // first of the wave's rows past the volume
    float* ldsf = reinterpret_cast<float*>(lds);
    // rows past the volume (the last block)
    for (int q = max(q0, qe); q < q1; ++q)
        for (int i = lane; i < nx; i += 64) ldsf[2 * ((q >> 1) * nx + i) + (q & 1)] = 0.0f;
    if (q0 >= qe) return;
    const int k0 = (row0 + q0) / ny, j0 = row0 + q0 - k0 * ny;
    for (int c0 = 0; c0 < nx;) {
        const int hl = c0 > 0 ? 1 : 0;                          // halo lane on the left
        const bool last = nx - c0 <= (64 - hl) * VW;            // no halo lane on the right
        const int c = c0 + VW * (lane - hl);                    // the lane's first column
        const bool own = lane >= hl && (last || lane < 63) && c < nx;
        const unsigned cu = (unsigned)min(c, nx - 1) & (kMaxLen - 1);  // (a bound the compiler sees)
        const int el = nx - 1 - c;                              // element that is the row's last column
        auto load = [&](Row& R, int r, int k) {
            const int dzp = (k + 1 < nz) ? nxy : nxy - N, dzm = (k > 0) ? -nxy : N - nxy;
            const QSM_GLOBAL float* xr = x + r * nx;
            const QSM_GLOBAL float* ur = u + r * nx;
            R.xc = ldu<VW>(xr + cu);
            R.ux = ldu<VW, NT>(ur + cu);
            R.uy = ldu<VW, NT>(ur + N + cu);
            R.uz = ldu<VW>(ur + 2 * N + cu);
            R.xzp = ldu<VW>(xr + dzp + cu);
            R.xzm = ldu<VW>(xr + dzm + cu);
            R.uzm = ldu<VW>(ur + 2 * N + dzm + cu);
            R.x0 = xr[0];
            R.xl = xr[nx - 1];
            R.ul = ur[nx - 1];
        };
        int j = j0, k = k0;
        Row A, B;
        FloatsU<VW> hx_m, hu_m, hx_p;  // rows above / below the wave's rows
        {
            const int r = row0 + q0, ra = j > 0 ? r - 1 : r + ny - 1;
            load(A, r, k);
            hx_m = ldu<VW>(x + ra * nx + cu);
            hu_m = ldu<VW>(u + N + ra * nx + cu);
        }
        float gym[VW];  // g's y component at y - 1
        auto gy_from = [&](const FloatsU<VW>& xc, const FloatsU<VW>& xm, const FloatsU<VW>& um) {
#pragma unroll
            for (int e = 0; e < VW; ++e) gym[e] = tv_gv((xc.v[e] - xm.v[e]) * hy + um.v[e], t);
        };
        // row q from cur, the next row's loads into nxt
        auto step = [&](const Row& cur, Row& nxt, int q) {
            const int r = row0 + q;
            int jn = j + 1, kn = k;
            if (jn == ny) {
                jn = 0;
                ++kn;
            }
            const bool more = q + 1 < qe;
            if (more) load(nxt, r + 1, kn);
            if (q + 2 >= qe) {  // the row after the wave's last row (or after this one), periodic in y
                const int rl = more ? r + 1 : r, jl = more ? jn : j;
                if (q + 2 == qe || q == q0) hx_p = ldu<VW>(x + (jl + 1 < ny ? rl + 1 : rl - ny + 1) * nx + cu);
            }
            if (q == q0) {
                gy_from(cur.xc, hx_m, hu_m);
            } else if (j == 0) {
                const int ra = r + ny - 1;
                gy_from(cur.xc, ldu<VW>(x + ra * nx + cu), ldu<VW>(u + N + ra * nx + cu));
            }
            FloatsU<VW> xyp;
            if (!more) xyp = hx_p;
            else if (jn == 0) xyp = ldu<VW>(x + (r - ny + 1) * nx + cu);
            else xyp = nxt.xc;
            const float rn = lane_next(cur.xc.v[0]);
            float ox[VW], oy[VW], oz[VW], gx[VW], gy[VW], d[VW];
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                float xp = e + 1 < VW ? cur.xc.v[e + 1 < VW ? e + 1 : 0] : rn;
                xp = el == e ? cur.x0 : xp;
                const float vx = (xp - cur.xc.v[e]) * hx + cur.ux.v[e];
                ox[e] = tv_clamp(vx, t);
                gx[e] = tv_g(vx, ox[e]);
            }
            float gl = lane_prev(gx[VW - 1]);
            gl = c == 0 ? tv_gv((cur.x0 - cur.xl) * hx + cur.ul, t) : gl;
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const float xc = cur.xc.v[e];
                const float vy = (xyp.v[e] - xc) * hy + cur.uy.v[e];
                const float vz = (cur.xzp.v[e] - xc) * hz + cur.uz.v[e];
                const float vzm = (xc - cur.xzm.v[e]) * hz + cur.uzm.v[e];
                oy[e] = tv_clamp(vy, t);
                oz[e] = tv_clamp(vz, t);
                gy[e] = tv_g(vy, oy[e]);
                // (the products' rounding is spelled out: the copies of this row
                // step, of which a row takes either by the rows of its block,
                // contracted the sum differently)
                const float dx = gx[e] - (e > 0 ? gx[e > 0 ? e - 1 : 0] : gl), dy = gy[e] - gym[e];
                d[e] = fmaf(tv_g(vz, oz[e]) - tv_gv(vzm, t), hz, fmaf(dx, hx, dy * hy));
                gym[e] = gy[e];
            }
            if (own) {
                QSM_GLOBAL float* o = uo + r * nx + cu;
                float* l = ldsf + 2 * ((q >> 1) * nx + c) + (q & 1);
                if (el >= VW - 1) {
                    stu<VW, NT>(o, ox);
                    stu<VW, NT>(o + N, oy);
                    stu<VW, NT>(o + 2 * N, oz);
#pragma unroll
                    for (int e = 0; e < VW; ++e) l[2 * e] = d[e];
                } else {
#pragma unroll
                    for (int e = 0; e < VW - 1; ++e) {
                        if (e <= el) {
                            o[e] = ox[e];
                            (o + N)[e] = oy[e];
                            (o + 2 * N)[e] = oz[e];
                            l[2 * e] = d[e];
                        }
                    }
                }
            }
            j = jn;
            k = kn;
        };
        int q = q0;
        for (; q + 1 < qe; q += 2) {
            step(A, B, q);
            step(B, A, q + 1);
        }
        if (q < qe) step(A, B, q);
        c0 += (64 - hl - (last ? 0 : 1)) * VW;
    }
}

// Columns per lane of fill_tvdiv_any: rows up to 256 columns in one group.
template <bool NT>
__device__ __forceinline__ void fill_tvdiv_runtime(float2* lds, const VolDesc& V, int nx, int RB, int row0, int nrows,
                                                   const QSM_GLOBAL float* __restrict__ x,
                                                   const QSM_GLOBAL float* __restrict__ u,
                                                   QSM_GLOBAL float* __restrict__ uo) {
    if (nx <= 64) fill_tvdiv_any<1, NT>(lds, V, nx, RB, row0, nrows, x, u, uo);
    else if (nx <= 128) fill_tvdiv_any<2, NT>(lds, V, nx, RB, row0, nrows, x, u, uo);
    else fill_tvdiv_any<4, NT>(lds, V, nx, RB, row0, nrows, x, u, uo);
}

// First step of an NLTV Newton round after the first (src/inversion/
// nltv.rs:86-120): the previous round ended either at convergence (no z/u
// update) or after max_iter steps (a z/u update with the previous weights is
// still due); then g was overwritten with grad(x).  So: u' = u or
// v - shrink(v, t w_old) with v = grad x + u, and the divergence source is
// bdiv(grad x).
template <int EMAX, bool RT>
__device__ __forceinline__ void fill_nltv_boundary(float2* lds, const VolDesc& V, int nx, int RB,
                                                   const QSM_GLOBAL float* __restrict__ x,
                                                   const QSM_GLOBAL float* __restrict__ u,
                                                   QSM_GLOBAL float* __restrict__ uo, int row0,
                                                   int nrows, bool converged,
                                                   const QSM_GLOBAL float* __restrict__ w, float wnorm) {
    const int ny = V.ny, nz = V.nz;
    const int nxy = nx * ny, N = nxy * nz;
    const float t = V.thr, hx = V.hx, hy = V.hy, hz = V.hz;
    const int total = RB * nx;
#pragma unroll
    for (int tt = 0; tt < EMAX; ++tt) {
        if (RT && tt * kThreads >= total) break;
        const int e = threadIdx.x + tt * kThreads;
        const int p = e / nx;
        const int i = e - p * nx;
        float d[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = row0 + 2 * p + h;
            const bool ok = (e < total) && (r < nrows);
            const int rr = ok ? r : 0;
            const int ii = ok ? i : 0;
            const int k = (int)fastdiv((uint32_t)rr, V.m_ny);
            const int j = rr - k * ny;
            const int idx = ii + rr * nx;
            const int dxp = (ii + 1 < nx) ? 1 : 1 - nx;
            const int dxm = (ii > 0) ? -1 : nx - 1;
            const int dyp = (j + 1 < ny) ? nx : nx - nxy;
            const int dym = (j > 0) ? -nx : nxy - nx;
            const int dzp = (k + 1 < nz) ? nxy : nxy - N;
            const int dzm = (k > 0) ? -nxy : N - nxy;
            const float xc = x[idx];
            const float gx = (x[idx + dxp] - xc) * hx, gy = (x[idx + dyp] - xc) * hy, gz = (x[idx + dzp] - xc) * hz;
            const float gxm = (xc - x[idx + dxm]) * hx, gym = (xc - x[idx + dym]) * hy, gzm = (xc - x[idx + dzm]) * hz;
            const float ux = u[idx], uy = u[N + idx], uz = u[2 * N + idx];
            if (ok) {
                if (converged) {
                    uo[idx] = ux;
                    uo[N + idx] = uy;
                    uo[2 * N + idx] = uz;
                } else {
                    const float ti = t * (w[idx] / wnorm);
                    const float vx = gx + ux, vy = gy + uy, vz = gz + uz;
                    uo[idx] = vx - shrinkf(vx, ti);
                    uo[N + idx] = vy - shrinkf(vy, ti);
                    uo[2 * N + idx] = vz - shrinkf(vz, ti);
                }
            }
            d[h] = ok ? (gx - gxm) * hx + (gy - gym) * hy + (gz - gzm) * hz : 0.0f;
        }
        if (e < total) lds[e] = make_float2(d[0], d[1]);
    }
}

// Adjoint of one unrolled TV-ADMM iteration, fused in front of the R2C of
// x-bar.  Forward iteration j (tol = 0, src/inversion/admm.rs:76-145):
//   c_j = bdiv(z_{j-1} - u_{j-1}),  x_j = A f - rho M c_j,
//   v_j = grad(x_j) + u_{j-1},  z_j = shrink(v_j, t),  u_j = v_j - z_j,
// with A = Re IFFT(D inv_a FFT .), M = Re IFFT(inv_a FFT .) (both
// symmetric) and t = lambda / rho.  Given c-bar_{j+1} = -rho M x-bar_{j+1}
// and s-bar_{j+1} (the adjoint of v_{j+1}), with q_j = sign(v_j) [|v_j| > t]:
//   z-bar_j = -grad c-bar_{j+1},  u-bar_j = s-bar_{j+1} + grad c-bar_{j+1},
//   s-bar_j = |q_j| z-bar_j + (1 - |q_j|) u-bar_j,
//   x-bar_j = grad^T s-bar_j = -bdiv(s-bar_j),
//   t-bar  += sum (u-bar_j - z-bar_j) q_j.
// The components of s-bar at i - e_a (needed by bdiv) are recomputed from
// c-bar, s-bar_{j+1} and q_j at i - e_a.  x-bar_j is added to the
// accumulator (field-bar = A sum_j x-bar_j); t-bar's FP64 partial is
// returned to the caller.  FIRST (j = K): x-bar_K = mask * chi-bar (chi = the
// masked x_K, src/utils/mask.rs:47-53), s-bar_K = 0.
__device__ __forceinline__ float adj_sbar(float g, float so, int8_t q) {
    return q != 0 ? -g : so + g;
}

template <int EMAX, bool FIRST, bool RT>
__device__ __forceinline__ void fill_tvadj(float2* lds, const VolDesc& V, int nx, int RB, int row0,
                                           int nrows, int ck, int par, double& tsum) {
    const int ny = V.ny, nz = V.nz;
    const int nxy = nx * ny, N = nxy * nz;
    const float hx = V.hx, hy = V.hy, hz = V.hz;
    const QSM_GLOBAL float* __restrict__ c = glb(V.adj_c);
    const QSM_GLOBAL float* __restrict__ so = glb(V.adj_s[par ^ 1]);
    QSM_GLOBAL float* __restrict__ sn = glb(V.adj_s[par]);
    const QSM_GLOBAL int8_t* __restrict__ q = glb(V.ckpt) + (size_t)(ck < 0 ? 0 : ck) * 3 * N;
    QSM_GLOBAL float* __restrict__ acc = glb(V.adj_acc);
    const int total = RB * nx;
    tsum = 0.0;
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        if (RT && t * kThreads >= total) break;
        const int e = threadIdx.x + t * kThreads;
        const int p = e / nx;
        const int i = e - p * nx;
        float d[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = row0 + 2 * p + h;
            const bool ok = (e < total) && (r < nrows);
            const int rr = ok ? r : 0;
            const int ii = ok ? i : 0;
            const int idx = ii + rr * nx;
            float xb;
            if constexpr (FIRST) {
                xb = (ok && glb(V.mask)[idx]) ? (float)glb(V.adj_chibar)[idx] : 0.0f;
                if (ok) {
                    sn[idx] = 0.0f;
                    sn[N + idx] = 0.0f;
                    sn[2 * N + idx] = 0.0f;
                    acc[idx] = xb;
                }
            } else {
                const int k = (int)fastdiv((uint32_t)rr, V.m_ny);
                const int j = rr - k * ny;
                const int dxp = (ii + 1 < nx) ? 1 : 1 - nx;
                const int dxm = (ii > 0) ? -1 : nx - 1;
                const int dyp = (j + 1 < ny) ? nx : nx - nxy;
                const int dym = (j > 0) ? -nx : nxy - nx;
                const int dzp = (k + 1 < nz) ? nxy : nxy - N;
                const int dzm = (k > 0) ? -nxy : N - nxy;
                const float cc = c[idx];
                const float cxp = c[idx + dxp], cyp = c[idx + dyp], czp = c[idx + dzp];
                const float cxm = c[idx + dxm], cym = c[idx + dym], czm = c[idx + dzm];
                const float sox = so[idx], soy = so[N + idx], soz = so[2 * N + idx];
                const float soxm = so[idx + dxm], soym = so[N + idx + dym], sozm = so[2 * N + idx + dzm];
                const int8_t qx = q[idx], qy = q[N + idx], qz = q[2 * N + idx];
                const int8_t qxm = q[idx + dxm], qym = q[N + idx + dym], qzm = q[2 * N + idx + dzm];
                const float gx = (cxp - cc) * hx, gy = (cyp - cc) * hy, gz = (czp - cc) * hz;
                const float gxm = (cc - cxm) * hx, gym = (cc - cym) * hy, gzm = (cc - czm) * hz;
                const float sx = adj_sbar(gx, sox, qx), sy = adj_sbar(gy, soy, qy), sz = adj_sbar(gz, soz, qz);
                const float sxm = adj_sbar(gxm, soxm, qxm), sym = adj_sbar(gym, soym, qym),
                            szm = adj_sbar(gzm, sozm, qzm);
                xb = -((sx - sxm) * hx + (sy - sym) * hy + (sz - szm) * hz);
                if (ok) {
                    sn[idx] = sx;
                    sn[N + idx] = sy;
                    sn[2 * N + idx] = sz;
                    acc[idx] += xb;
                    tsum += (double)(sox + 2.0f * gx) * (double)qx + (double)(soy + 2.0f * gy) * (double)qy +
                            (double)(soz + 2.0f * gz) * (double)qz;
                } else {
                    xb = 0.0f;
                }
            }
            d[h] = xb;
        }
        if (e < total) lds[e] = make_float2(d[0], d[1]);
    }
}

// ------------------------------------------------------------- R2C x pass --
// Row-block index of dispatch slot lb when every plane holds a whole number
// bpp = ny / R of R-row blocks: slots run plane-fastest (lb = yb nz + k), so
// blocks dispatched together (and sharing an XCD) hold the same rows of
// neighbouring planes, and the divergence's loads of x at k +- 1 and u_z at
// k - 1 find the rows their neighbours just read in L2.  Otherwise slots are
// blocks in row order.  A bijection on [0, bpp nz) either way.
__device__ __forceinline__ int plane_fast_block(int lb, int ny, int nz, int R) {
    const int bpp = ny / R;
    if (bpp * R != ny) return lb;
    const int yb = lb / nz;
    return (lb - yb * nz) * bpp + yb;
}

// Block = RB pairs of real rows.  Pair p packs rows (2p, 2p+1) as
// z = a + i b; after a complex FFT of length nx the half spectra are
//   A[k] = (Z[k] + conj Z[-k]) / 2,   B[k] = (Z[k] - conj Z[-k]) / (2i).
// aux: TV iteration parity for SRC_TVDIV, radius index for SRC_SPHERE.
// ck: checkpoint index (SRC_TVDIV_REC: the record written; SRC_TVADJ: the
// record read, and the row of adj_tpart written).
// RBS: the block takes shifted_rows(N, RBS) pair-rows (small volumes: more,
// smaller blocks); the host sizes rows_x and the launch the same way.
template <int N, int EG, int SRC, int RBS = 0, bool NT = false>
__global__ __launch_bounds__(kThreads) void k_r2c_x(const VolDesc* __restrict__ vols, LaunchTable lt,
                                                    const float2* __restrict__ tw, int out_sel, int aux,
                                                    const VolStatus* status, VolStatus* status_rw,
                                                    VolStatus* mirror, int ck) {
    constexpr int RBX = N > 0 ? qsmfft::shifted_rows(N, RBS) : 0;
    static_assert(N == 0 || RBX >= 1, "row shift too large for this length");
    constexpr int EMAX = N > 0 ? (RBX * N + kThreads - 1) / kThreads : x_emax(0, EG);
    __shared__ float2 lds[N > 0 ? RBX * N : x_lds(0, EG)];
    __shared__ float2 twl[tw_lds(N, EG)];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    if (status && status[gv].done) return;
    if constexpr (SRC == SRC_TVDIV || SRC == SRC_TVDIV_REC) {
        // The first block of a volume closes the previous iteration: it
        // reduces the C2R pass's sums and may mark the volume converged.
        // Blocks of this pass that still see it running do work that is
        // discarded (they write only the spectrum and the dual variable,
        // never the iterate x that is returned).
        __shared__ double sh[kThreads / 64];
        if (status_rw && lb == 0) tv_reduce_block(V, gv, status_rw, mirror, sh);
    }
    const int nx = N > 0 ? N : V.nx;
    const int nxh = (nx + 1) / 2;
    const int RB = N > 0 ? RBX : V.rows_x;
    const int nrows = V.ny * V.nz;
    const int rb = (SRC == SRC_TVDIV || SRC == SRC_TVDIV_REC || SRC == SRC_TVDIV_W || SRC == SRC_NLTV_BND)
                       ? plane_fast_block(lb, V.ny, V.nz, 2 * RB)
                       : lb;
    const int row0 = rb * RB * 2;
    TwStage<N, EG> tws;
    tws.fetch(tw, V.px);
    if constexpr (SRC == SRC_TVDIV && tvdiv_rows_form(N, RBX)) {
        fill_tvdiv_rows<N, RBX, NT>(lds, V, row0, nrows, glb(V.x[aux]), glb(V.u[aux ^ 1]), glb(V.u[aux]));
    } else if constexpr (SRC == SRC_TVDIV && N == 0 && eg_dense(EG)) {
        fill_tvdiv_runtime<NT>(lds, V, nx, RB, row0, nrows, glb(V.x[aux]), glb(V.u[aux ^ 1]), glb(V.u[aux]));
    } else if constexpr (SRC == SRC_TVDIV) {
        fill_tvdiv<EMAX, false, false, NT, N == 0>(lds, V, nx, RB, glb(V.x[aux]), glb(V.u[aux ^ 1]), glb(V.u[aux]),
                                                   row0, nrows, nullptr);
    } else if constexpr (SRC == SRC_TVDIV_REC) {
        const size_t N3 = (size_t)3 * V.nx * V.ny * V.nz;
        fill_tvdiv<EMAX, true, false, false, N == 0>(lds, V, nx, RB, glb(V.x[aux]), glb(V.u[aux ^ 1]), glb(V.u[aux]),
                                                     row0, nrows, glb(V.ckpt) + (size_t)ck * N3);
    } else if constexpr (SRC == SRC_TVDIV_W) {
        fill_tvdiv<EMAX, false, true, false, N == 0>(lds, V, nx, RB, glb(V.x[aux]), glb(V.u[aux ^ 1]), glb(V.u[aux]),
                                                     row0, nrows, nullptr, glb(V.nltv_w[ck]), (float)V.nltv_wnorm[ck]);
    } else if constexpr (SRC == SRC_NLTV_BND) {
        // status_rw carries the convergence state of the round just ended
        fill_nltv_boundary<EMAX, N == 0>(lds, V, nx, RB, glb(V.x[aux]), glb(V.u[aux ^ 1]), glb(V.u[aux]), row0,
                                 nrows, status_rw[gv].done != 0, glb(V.nltv_w[ck]),
                                 (float)V.nltv_wnorm[ck]);
    } else if constexpr (SRC == SRC_TVADJ_FIRST || SRC == SRC_TVADJ) {
        __shared__ double sh[kThreads / 64];
        double ts;
        fill_tvadj<EMAX, SRC == SRC_TVADJ_FIRST, N == 0>(lds, V, nx, RB, row0, nrows, ck, aux, ts);
        if constexpr (SRC == SRC_TVADJ) {
            const double bt = block_sum(ts, sh);
            if (threadIdx.x == 0) glb(V.adj_tpart)[(size_t)ck * V.adj_nblk + lb] = bt;
        }
    } else {
        fill_simple<N, EMAX, SRC>(lds, V, nx, RB, row0, nrows, aux);
    }
    tws.commit(twl);
    __syncthreads();
    run_fft<N, EG, EMAX, false, 0, false, RBX>(lds, V.px, RB, 1, nx, twl, tw);
    QSM_GLOBAL float2* __restrict__ out = glb(V.spec[out_sel]);
    const int total = RB * nxh;
    if constexpr (N > 0 && N % 4 == 0) {
        // two consecutive half-spectrum entries per thread and row: 16-byte
        // stores (nxh is even, so every pair is 16-byte aligned)
        constexpr int NH2 = N / 4, TOT2 = RBX * NH2;
#pragma unroll
        for (int t = 0; t < (TOT2 + kThreads - 1) / kThreads; ++t) {
            const int e = threadIdx.x + t * kThreads;
            if (e < TOT2) {
                const int p = e / NH2;
                const int k0 = 2 * (e - p * NH2);
                const int ra = row0 + 2 * p, rb = ra + 1;
                float a4[4], b4[4];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int k = k0 + c;
                    const float2 zk = lds[p * N + k];
                    const float2 zm = lds[p * N + (k == 0 ? 0 : N - k)];
                    float2 A = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
                    float2 B = make_float2(0.5f * (zk.y + zm.y), -0.5f * (zk.x - zm.x));
                    if (k == 0) {
                        // (DC, Nyquist) of both rows: real parts of Z[0] and Z[N/2]
                        const float2 zn = lds[p * N + N / 2];
                        A = make_float2(zk.x, zn.x);
                        B = make_float2(zk.y, zn.y);
                    }
                    a4[2 * c] = A.x;
                    a4[2 * c + 1] = A.y;
                    b4[2 * c] = B.x;
                    b4[2 * c + 1] = B.y;
                }
                if (ra < nrows) stv<4>((QSM_GLOBAL float*)(out + k0 + (size_t)ra * nxh), vpack<4>(a4));
                if (rb < nrows) stv<4>((QSM_GLOBAL float*)(out + k0 + (size_t)rb * nxh), vpack<4>(b4));
            }
        }
        return;
    }
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < total) {
            const int p = div_nxh<N>(e, V);
            const int k = e - p * nxh;
            const int ra = row0 + 2 * p, rb = ra + 1;
            const float2 zk = lds[p * nx + k];
            const float2 zm = lds[p * nx + (k == 0 ? 0 : nx - k)];
            float2 A = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
            float2 B = make_float2(0.5f * (zk.y + zm.y), -0.5f * (zk.x - zm.x));
            if ((nx & 1) == 0 && k == 0) {
                // (DC, Nyquist) of both rows: real parts of Z[0] and Z[nx/2]
                const float2 zn = lds[p * nx + nx / 2];
                A = make_float2(zk.x, zn.x);
                B = make_float2(zk.y, zn.y);
            }
            if (ra < nrows) stg2(out + k + (size_t)ra * nxh, A);
            if (rb < nrows) stg2(out + k + (size_t)rb * nxh, B);
        }
    }
}

// ------------------------------------------------------------- C2C y pass --
// Block = one tile of TW consecutive kx columns at one kz, full ny (TW =
// kTile; kTileLong for runtime-planned lengths above 256).
// sel2 >= 0 transforms a second spectrum with a second set of blocks.
// SCHED 0: two-stage column FFT (fft_col2.hpp) where the length allows;
// SCHED 1: the LDS-staged Stockham stages (less LDS per block).
template <int N, int EG, bool INV, int SCHED, int TW = kTile>
__global__ __launch_bounds__(kThreads) void k_y_pass(const VolDesc* __restrict__ vols, LaunchTable lt,
                                                     const float2* __restrict__ tw, int sel, int sel2,
                                                     const VolStatus* __restrict__ status) {
    static_assert(TW == kTile || N == 0, "compiled lengths use tiles of kTile columns");
    constexpr int EMAX = col_emax(N, EG);
    constexpr bool TWO = SCHED == 0 && qsmfft::col2_ok(N);
    __shared__ float2 lds[TWO ? col_lds2(N, EG) : col_lds(N, EG)];
    __shared__ float2 twl[tw_lds(N, EG)];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    if (status && status[gv].done) return;
    const int ntx = TW == kTile ? V.ntx : V.ntx_long;
    const int per = ntx * V.nz;
    int s = sel;
    if (lb >= per) { lb -= per; s = sel2; }
    const int kz = lb / ntx;
    const int tx = lb - kz * ntx;
    const int kx0 = tx * TW;
    const int nxh = V.nxh;
    const int ny = N > 0 ? N : V.ny;
    QSM_GLOBAL float2* buf = glb(V.spec[s]) + (size_t)kz * nxh * ny;
    TwStage<N, EG> tws;
    tws.fetch(tw, V.py);
    // tile 0 of an even-nx volume: column 0 is packed (DC and Nyquist planes)
    const bool pkc = tx == 0 && packed_x(V);
    if constexpr (TWO) {
        constexpr int R0 = N / 16;
        const int c = threadIdx.x & 15, j = threadIdx.x >> 4;
        float2 v[16];
        l16_load<R0>(v, buf, nxh, kx0, nxh);
        tws.commit(twl);
        // column 0 of a packed tile goes through LDS (free before the
        // first exchange and after the last one)
        if constexpr (INV) {
            if (pkc) {  // L16 layout: thread (j, c) holds rows j + 16 r
                if (c == 0) {
#pragma unroll
                    for (int r = 0; r < R0; ++r) lds[j + 16 * r] = v[r];
                }
                __syncthreads();
                if (c == 0) {
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int row = j + 16 * r;
                        v[r] = ypk_inv(row, N, v[r], lds[mirror_idx(row, N)]);
                    }
                }
                __syncthreads();  // before the transform's first exchange writes
            }
        }
        qsmfft::Col2<R0>::template l16_to_lr<INV>(v, lds, twl);
        if constexpr (!INV) {
            if (pkc) {  // LR layout: thread (j < R0, c) holds rows j + R0 r
                __syncthreads();  // the transform's last reads are done
                if (c == 0 && j < R0) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) lds[j + R0 * r] = v[r];
                }
                __syncthreads();
                if (c == 0 && j < R0) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int row = j + R0 * r;
                        v[r] = ypk_fwd(row, N, v[r], lds[mirror_idx(row, N)]);
                    }
                }
            }
        }
        lr_store<R0>(v, buf, nxh, kx0, nxh);
    } else {
        col_load<EMAX, TW>(lds, buf, nxh, ny, kx0, nxh);
        tws.commit(twl);
        __syncthreads();
        if (INV && pkc) ypk_lds<true, TW>(lds, ny);
        run_fft<N, EG, EMAX, true, tile_log2(TW), INV>(lds, V.py, TW, TW, 1, twl, tw);
        if (!INV && pkc) ypk_lds<false, TW>(lds, ny);
        col_store<EMAX, TW>(lds, buf, nxh, ny, kx0, nxh);
    }
}

// ---------------------------------------------------- TV spectral passes --
// The periodic second difference along one axis, (2 - 2 cos(2 pi k / n)) /
// vs^2: the Poisson eigenvalue of src/unwrap/laplacian.rs:93-118 (negated),
// 0 at k = 0 and on every length-1 axis.
__device__ inline double lap_closed(int k, int n, double vs) {
#pragma clang fp contract(off)
    const double two_pi = 6.283185307179586476925286766559;
    return (2.0 - 2.0 * cos(two_pi * k / n)) / (vs * vs);
}

// One axis's share of the DFT of the negative Laplacian stencil of
// src/kernels/laplacian.rs:20-62.  That stencil is written by assignment:
// the centre holds 2/vs^2 for every axis, the two neighbours -1/vs^2 only
// where n > 1, and where n = 2 both neighbours are the same voxel, written
// once.  So the share is the periodic second difference where n > 2, but
// 2/vs^2 (at every k, DC included) where n = 1 and (2 - cos(pi k))/vs^2,
// i.e. 1/vs^2 at k = 0 and 3/vs^2 at k = 1, where n = 2.
__device__ inline double lap_stencil(int k, int n, double vs) {
#pragma clang fp contract(off)
    if (n > 2) return lap_closed(k, n, vs);
    return (n == 1 ? 2.0 : (k == 0 ? 1.0 : 3.0)) / (vs * vs);
}

// Spectral terms in FP64 with every operation rounded (no contraction) so
// threshold decisions match the reference's f64 arithmetic:
// D = 1/3 - (k.b)^2/|k|^2, 0 where |k|^2 <= 1e-20 (src/kernels/dipole.rs:
// 24-72), and L, the DFT of the negative Laplacian stencil (lap_stencil per
// axis; exactly 0 at DC unless an axis has length 1).
//
// Every sum runs over x, y, then z, so the x and y parts are formed once per
// column (a thread's elements of a z tile share it) and the z part of L, a
// cosine, once per block into a table.  Formed per element, the six cosines
// of an index and its mirror bound these passes: 90.5 us for the TKD z pass
// at 192x192x128 (0.8 TB/s), 145 / 118 us for the two RTS ones at
// 224x224x144.  The values are the same, bit for bit.

// One axis's share of L: lap_stencil, lap_closed (the Poisson filter), or
// none where the multiplier does not use L.
enum LapKind : int { LAP_NONE = 0, LAP_STENCIL = 1, LAP_CLOSED = 2 };
__device__ inline double lap_axis(int kind, int k, int n, double vs) {
    return kind == LAP_STENCIL ? lap_stencil(k, n, vs) : (kind == LAP_CLOSED ? lap_closed(k, n, vs) : 0.0);
}

// (D, L) at an index and at its mirror.
struct SpecPair {
    double D, L, Dm, Lm;
};

// The x and y parts of one column (kx, ky) and of its mirror.
struct SpecXY {
    double s, sm;    // fx bx + fy by
    double k2;       // fx^2 + fy^2 (the same for the mirror: its f are +-f)
    double l, lm;    // the x and y shares of L
    double dfz, bz;  // fftfreq step along z, z component of B0
    __device__ void init(const VolDesc& V, int kx, int ky, int lap) {
#pragma clang fp contract(off)
        const int mx = mirror_idx(kx, V.nx), my = mirror_idx(ky, V.ny);
        const double fx = fftfreq_at(kx, V.nx, V.vsx), fy = fftfreq_at(ky, V.ny, V.vsy);
        const double fxm = fftfreq_at(mx, V.nx, V.vsx), fym = fftfreq_at(my, V.ny, V.vsy);
        s = fx * V.bx + fy * V.by;
        sm = fxm * V.bx + fym * V.by;
        k2 = fx * fx + fy * fy;
        l = lap_axis(lap, kx, V.nx, V.vsx) + lap_axis(lap, ky, V.ny, V.vsy);
        lm = lap_axis(lap, mx, V.nx, V.vsx) + lap_axis(lap, my, V.ny, V.vsy);
        dfz = 1.0 / ((double)V.nz * V.vsz);
        bz = V.bz;
    }
    // lz: the block's table of z shares (lap_axis at every kz)
    __device__ __forceinline__ SpecPair at(int kz, int nz, const double* lz) const {
#pragma clang fp contract(off)
        const int mz = mirror_idx(kz, nz);
        const double fz = (double)(kz < (nz + 1) / 2 ? kz : kz - nz) * dfz;
        const double fzm = (double)(mz < (nz + 1) / 2 ? mz : mz - nz) * dfz;
        const double kdb = s + fz * bz, kdbm = sm + fzm * bz;
        const double q2 = k2 + fz * fz;
        const double kk = kdb * kdb, kkm = kdbm * kdbm;
        SpecPair p;
        p.D = (q2 > 1e-20) ? (1.0 / 3.0) - kk / q2 : 0.0;
        // the mirror's k.b is -k.b but on Nyquist planes
        p.Dm = kkm == kk ? p.D : ((q2 > 1e-20) ? (1.0 / 3.0) - kkm / q2 : 0.0);
        p.L = lz ? l + lz[kz] : 0.0;
        p.Lm = lz ? lm + lz[mz] : 0.0;
        return p;
    }
};

// TV: D inv_a and inv_a, inv_a = 1/(D^2 + rho L) or 0 where |.| <= 1e-20
// (src/inversion/admm.rs:157-168).
__device__ inline void tv_multipliers(const VolDesc& V, double D, double L, double& dinv, double& inv) {
#pragma clang fp contract(off)
    const double a = D * D + V.rho * L;
    inv = (fabs(a) > 1e-20) ? 1.0 / a : 0.0;
    dinv = D * inv;
}

// RTS (src/inversion/rts.rs:102-183): M = mu on the cone |D| > delta, else 0;
// inv_a = rho / (M + rho L) or 0; f^ multiplier (M / rho) inv_a where both
// are non-zero; the ADMM step uses rho = 1, so its multiplier is inv_a.
__device__ inline void rts_multipliers(const VolDesc& V, double D, double L, double& fm, double& inv) {
#pragma clang fp contract(off)
    const double M = (fabs(D) > V.filt_a) ? V.filt_b : 0.0;
    const double a = M + V.rho * L;
    inv = (fabs(a) > 1e-20) ? V.rho / a : 0.0;
    fm = (fabs(M) > 1e-20 && fabs(inv) > 1e-20) ? (M / V.rho) * inv : 0.0;
}

// Closed-form spectral inversions, one multiplier per frequency:
//   TKD  1/D, or sign(D)/thr where |D| <= thr      (src/inversion/tkd.rs:48-99)
//   TSVD 1/D, or 0 where |D| <= thr                 (the tsvd after it)
//   Tikhonov D / (D^2 + lambda Gamma), Gamma = 1, L or L^2, 0 where the
//     denominator is <= 1e-20                        (src/inversion/tikhonov.rs:62-131)
//   RTS step 1: lsmr_iter rounds of w += (1 - w D) D/(D^2 + 1e-6) from
//     w = D/(D^2 + 1e-6) on the cone |D| > delta, 0 off it (the per-frequency
//     refinement of src/inversion/rts.rs:117-150, applied to FFT(f))
//   Poisson: 1/lambda with lambda the periodic Laplacian's eigenvalue
//     (lap_closed summed over the axes, negated), 0
//     where |lambda| <= 1e-20 (src/unwrap/laplacian.rs:93-133)
enum Filter : int { FILT_TKD = 0, FILT_TSVD = 1, FILT_TIK_ID = 2, FILT_TIK_GRAD = 3, FILT_TIK_LAP = 4,
                    FILT_RTS_X0 = 5, FILT_POISSON = 6 };

__device__ inline double filter_mult(const VolDesc& V, double D, double L) {
#pragma clang fp contract(off)
    const double p = V.filt_a;
    switch (V.filt) {
        case FILT_TKD: {
            const double inv_t = 1.0 / p;
            return fabs(D) <= p ? (D >= 0.0 ? inv_t : -inv_t) : 1.0 / D;
        }
        case FILT_TSVD: return fabs(D) <= p ? 0.0 : 1.0 / D;
        case FILT_TIK_ID:
        case FILT_TIK_GRAD:
        case FILT_TIK_LAP: {
            const double g = V.filt == FILT_TIK_ID ? 1.0 : (V.filt == FILT_TIK_GRAD ? L : L * L);
            const double denom = D * D + p * g;
            return fabs(denom) > 1e-20 ? D / denom : 0.0;
        }
        case FILT_POISSON: {
            const double lam = -L;
            return fabs(lam) > 1e-20 ? 1.0 / lam : 0.0;
        }
        default: {  // FILT_RTS_X0
            if (!(fabs(D) > p)) return 0.0;
            const double gk = D / (D * D + 1e-6);
            double w = gk;
            for (int it = 0; it < V.lsmr_iter; ++it) w += (1.0 - w * D) * gk;
            return w;
        }
    }
}

enum ZOp : int {
    ZOP_TV_SETUP = 0, ZOP_TV_SOLVE = 1, ZOP_VS_FWD = 2, ZOP_VS_RADIUS = 3, ZOP_VS_DECONV = 4,
    ZOP_TV_ADJ = 5,     // c-bar^ = -rho inv_a x-bar^ / N (the adjoint of the x-update in c)
    ZOP_TV_APPLYA = 6,  // field-bar^ = D inv_a acc^ / N  (the adjoint in f, A is symmetric)
    ZOP_DIPOLE = 7,     // D chi^ / N  (the dipole forward operator, self-adjoint)
    ZOP_FILTER = 8,     // closed-form inversion multiplier / N (filter_mult)
    ZOP_RTS_SETUP = 9,  // as TV_SETUP with the RTS multipliers
    ZOP_TV_SOLVE0 = 10, // first ADMM step from g = 0: x^ = f^, inverse z only
    ZOP_RTS_SOLVE = 11  // ZOP_TV_SOLVE with the stored multiplier q (RTS)
};

// The TV x-update multiplier q = rho inv_a / N, inv_a = 1/(D^2 + rho L) (0 at
// DC; src/inversion/admm.rs:157-168), averaged over k and its mirror as the
// stored one is, formed in FP32 where it is used instead of being read (it
// is the same at every iteration; reading it costs 4 bytes per spectral
// element per iteration).  There is no threshold in it besides DC, so FP32
// only perturbs it by a few ulp.  k and its mirror differ only on Nyquist
// planes, where the mirror keeps the (negative) Nyquist frequency.
// init: the x and y terms of one column (FP64, once per thread); at: one kz,
// with twz = exp(-2 pi i kz / nz) from the z pass's twiddle table.
struct TvQ {
    float sxy, sxym, k2xy, lxy, rlxy, dfz, bz, hz2, rho, scale;
    bool sym;  // the mirror of (kx, ky) is (-kx, -ky): no Nyquist index in it
    // In FP32 (the multiplier is FP32): fftfreq (src/fft.rs:544-566), whose
    // mirror is its negative except at a Nyquist index, and lap_stencil with
    // 2 - 2 cos t written as 4 sin^2(t / 2) (no cancellation).
    __device__ __forceinline__ void init(const VolDesc& V, int kx, int ky) {
        const bool nyx = 2 * kx == V.nx, nyy = 2 * ky == V.ny;
        sym = !nyx && !nyy;
        // 1/(n vs) and 1/vs^2 from the FP32 1/vs (V.hx ...)
        const float fx = (float)(kx < (V.nx + 1) / 2 ? kx : kx - V.nx) * (V.hx * __builtin_amdgcn_rcpf((float)V.nx));
        const float fy = (float)(ky < (V.ny + 1) / 2 ? ky : ky - V.ny) * (V.hy * __builtin_amdgcn_rcpf((float)V.ny));
        const float fxm = nyx ? fx : -fx, fym = nyy ? fy : -fy;
        const float bx = (float)V.bx, by = (float)V.by;
        sxy = fx * bx + fy * by;
        sxym = fxm * bx + fym * by;
        k2xy = fx * fx + fy * fy;
        auto lap = [](int k, int n, float h) {
            const float h2 = h * h;
            if (n > 2) {
                const float sn = sinpif((float)k / (float)n);
                return 4.0f * (sn * sn) * h2;
            }
            return (n == 1 ? 2.0f : (k == 0 ? 1.0f : 3.0f)) * h2;
        };
        lxy = lap(kx, V.nx, V.hx) + lap(ky, V.ny, V.hy);
        rho = (float)V.rho;
        rlxy = rho * lxy;
        dfz = V.hz * __builtin_amdgcn_rcpf((float)V.nz);
        bz = (float)V.bz;
        hz2 = V.hz * V.hz;
        scale = 0.5f * rho * __builtin_amdgcn_rcpf((float)V.nx * (float)V.ny * (float)V.nz);
    }
    __device__ __forceinline__ float at(int kz, int nz, float2 twz) const {
        const int sz = kz < (nz + 1) / 2 ? kz : kz - nz;           // fftfreq index
        const int szm = (2 * kz == nz) ? sz : -sz;                  // its mirror's
        const float fz = (float)sz * dfz, fzm = (float)szm * dfz;
        const float kdb = sxy + fz * bz, kdbm = sxym + fzm * bz;
        const float k2 = k2xy + fz * fz;
        // 2 - 2 cos(t) = 2 sin^2(t) / (1 + cos(t)) where cos(t) > 0 (no
        // cancellation); lap_stencil's shares where nz <= 2 (twz.x = cos(pi kz)
        // where nz = 2)
        const float cz = twz.x;
        const float lz = (nz > 2 ? (cz > 0.0f ? 2.0f * (twz.y * twz.y) * __builtin_amdgcn_rcpf(1.0f + cz)
                                              : 2.0f - 2.0f * cz)
                                 : (nz == 1 ? 2.0f : 2.0f - cz)) * hz2;
        const float rl = rho * (lxy + lz);
        const float rk = k2 > 1e-20f ? __builtin_amdgcn_rcpf(k2) : 0.0f;  // D = 0 at DC
        const float D = k2 > 1e-20f ? (1.0f / 3.0f) - kdb * kdb * rk : 0.0f;
        const float a = D * D + rl;
        const float ia = a > 1e-20f ? __builtin_amdgcn_rcpf(a) : 0.0f;
        // where the mirror is -k (sym, kz not the Nyquist plane) sxym = -sxy
        // and fzm = -fz exactly, so kdbm = -kdb and its term is ia bit for bit
        if (sym && 2 * kz != nz) return scale * (ia + ia);
        const float Dm = k2 > 1e-20f ? (1.0f / 3.0f) - kdbm * kdbm * rk : 0.0f;
        const float am = Dm * Dm + rl;
        const float iam = am > 1e-20f ? __builtin_amdgcn_rcpf(am) : 0.0f;
        return scale * (ia + iam);
    }
    // The terms of at() that depend on kz only, shared by every column of a
    // z tile: (fz bz, fz^2, rho lz / vs_z^2) with fz the plane's frequency
    // and lz its share of the Laplacian (cos and sin of 2 pi kz / nz here).
    __device__ static float4 plane(const VolDesc& V, int kz, int nz) {
        const float dfz = V.hz * __builtin_amdgcn_rcpf((float)nz);
        const int sz = kz < (nz + 1) / 2 ? kz : kz - nz;
        const float fz = (float)sz * dfz;
        float sn, cs;
        sincospif(2.0f * (float)kz / (float)nz, &sn, &cs);
        const float lz = (nz > 2 ? (cs > 0.0f ? 2.0f * (sn * sn) * __builtin_amdgcn_rcpf(1.0f + cs)
                                              : 2.0f - 2.0f * cs)
                                 : (nz == 1 ? 2.0f : 2.0f - cs)) *
                         (V.hz * V.hz);
        return make_float4(fz * (float)V.bz, fz * fz, (float)V.rho * lz, 0.0f);
    }
    // at() from the plane's terms P = plane(V, kz, nz)
    __device__ __forceinline__ float at_plane(int kz, int nz, float4 P) const {
        const float kdb = sxy + P.x;
        const float k2 = k2xy + P.y;
        const float rl = rlxy + P.z;
        const float rk = k2 > 1e-20f ? __builtin_amdgcn_rcpf(k2) : 0.0f;  // D = 0 at DC
        const float D = k2 > 1e-20f ? (1.0f / 3.0f) - kdb * kdb * rk : 0.0f;
        const float a = D * D + rl;
        const float ia = a > 1e-20f ? __builtin_amdgcn_rcpf(a) : 0.0f;
        if (sym && 2 * kz != nz) return scale * (ia + ia);
        const float kdbm = sxym + (2 * kz == nz ? P.x : -P.x);  // the mirror's kz is -kz but on Nyquist
        const float Dm = k2 > 1e-20f ? (1.0f / 3.0f) - kdbm * kdbm * rk : 0.0f;
        const float am = Dm * Dm + rl;
        const float iam = am > 1e-20f ? __builtin_amdgcn_rcpf(am) : 0.0f;
        return scale * (ia + iam);
    }
};

// The L that the multiplier of an FP64 z pass uses (block-uniform).
template <int OP>
__device__ __forceinline__ int lap_kind(const VolDesc& V) {
    if constexpr (OP == ZOP_DIPOLE) return LAP_NONE;
    else if constexpr (OP != ZOP_FILTER) return LAP_STENCIL;
    else
        return V.filt == FILT_POISSON ? LAP_CLOSED
                                      : (V.filt == FILT_TIK_GRAD || V.filt == FILT_TIK_LAP ? LAP_STENCIL : LAP_NONE);
}

// Symmetrised multipliers of the spectral setup at one frequency, averaged
// over k and its mirror (the reference keeps Re(IFFT(.)) of a full
// spectrum, the inverse of its Hermitian part; on Nyquist planes D(k) !=
// D(-k) when B0 is tilted): m for f^ and q = rho inv_a / N (TV) or
// inv_a / N (RTS).
template <int OP>
__device__ inline void setup_mult(const VolDesc& V, const SpecPair& p, double& m, double& qv) {
    const double invN = 1.0 / ((double)V.nx * V.ny * V.nz);
    double d1, i1, d2, i2;
    if constexpr (OP == ZOP_TV_SETUP) {
        tv_multipliers(V, p.D, p.L, d1, i1);
        tv_multipliers(V, p.Dm, p.Lm, d2, i2);
        m = 0.5 * (d1 + d2) * invN;
        qv = V.rho * 0.5 * (i1 + i2) * invN;
    } else {
        rts_multipliers(V, p.D, p.L, d1, i1);
        rts_multipliers(V, p.Dm, p.Lm, d2, i2);
        m = 0.5 * (d1 + d2) * invN;
        qv = 0.5 * (i1 + i2) * invN;
    }
}

// Symmetrised multiplier of APPLYA (D inv_a / N), DIPOLE (D / N) or FILTER.
template <int OP>
__device__ inline double apply_mult(const VolDesc& V, const SpecPair& p) {
    const double invN = 1.0 / ((double)V.nx * V.ny * V.nz);
    if constexpr (OP == ZOP_TV_APPLYA) {
        double d1, i1, d2, i2;
        tv_multipliers(V, p.D, p.L, d1, i1);
        tv_multipliers(V, p.Dm, p.Lm, d2, i2);
        return 0.5 * (d1 + d2) * invN;
    } else if constexpr (OP == ZOP_DIPOLE) {
        return 0.5 * (p.D + p.Dm) * invN;
    } else {
        const double m1 = filter_mult(V, p.D, p.L);
        const double m2 = (p.Dm == p.D && p.Lm == p.L) ? m1 : filter_mult(V, p.Dm, p.Lm);
        return 0.5 * (m1 + m2) * invN;
    }
}

// TV z pass.  SETUP: forward z of FFT(f) (after x, y), then
//   f^ = FFT(f) * D * inv_a / N  -> SPEC_A,   rho * inv_a / N -> q,
// with both multipliers averaged over k and -k: the reference keeps
// Re(IFFT(.)) of a full spectrum, which equals the inverse of its Hermitian
// part, and on Nyquist planes D(k) != D(-k) when B0 is tilted.
// SOLVE: forward z, x^ = f^ - q * FFT(div) (src/inversion/admm.rs:106-108,
// scaled by 1/N), inverse z, with q formed in-kernel (TvQ); RTS_SOLVE reads
// the stored q instead.  ADJ: forward z, -q * spectrum, inverse z (q from
// TvQ).  APPLYA / DIPOLE: forward z, times the Hermitian part of D inv_a / N
// or of D / N (in FP64), inverse z.
// The stored q of the Nyquist plane's half of the two doubly packed columns
// (ky = 0 and ny / 2, nz values each) follows the tile-major array.  (Formed
// in FP64 by the 16 threads of such a column at every RTS iteration instead,
// it held the whole z pass: 85 us at 224x224x144, 1.0 TB/s.)
__device__ __forceinline__ size_t q_nyq_base(const VolDesc& V, int ky) {
    return V.q_len + (ky == 0 ? 0 : (size_t)V.nz);
}
// The per-iteration ops (SOLVE, SOLVE0, ADJ, RTS_SOLVE) at the lengths of
// fft_col2.hpp: forward z from the load layout, the product in registers,
// inverse z back to the load layout; two LDS exchanges in all.
template <int N, int EG, int OP, bool NT>
__device__ __forceinline__ void z_tv_col2(const VolDesc& V, float2* lds, float2* twl, const TwStage<N, EG>& tws,
                                          int ky, int kx0, bool dpk) {
    constexpr int R0 = N / 16;
    using C = qsmfft::Col2<R0>;
    const int nxh = V.nxh;
    const size_t zs = (size_t)nxh * V.ny;
    const size_t base = (size_t)ky * nxh;
    QSM_GLOBAL float2* buf = glb(V.spec[SPEC_WORK]) + base;
    float2 v[16];
    if constexpr (OP == ZOP_TV_SOLVE0) {
        // g = 0 before the first step (AdmmBuffers::new), so div = 0 and x^ = f^
        l16_load<R0>(v, glb(V.spec[SPEC_A]) + zop_base(ky, kx0 / kTile, V.ntx, N, kTile), kTile, kx0, nxh);
        tws.commit(twl);
        C::template l16_to_lr<true>(v, lds, twl);
        lr_store<R0>(v, buf, zs, kx0, nxh);
        return;
    }
    l16_load<R0>(v, buf, zs, kx0, nxh);
    // x-update operands in the LR layout, in flight during the forward FFT
    const int c = threadIdx.x & 15, j = threadIdx.x >> 4;
    const bool act = j < R0;
    constexpr bool HAS_F = OP == ZOP_TV_SOLVE || OP == ZOP_RTS_SOLVE;
    constexpr bool Q_MEM = OP == ZOP_RTS_SOLVE;
    float2 fr[HAS_F ? 16 : 1];
    float qr[16];
    {
        // threads j >= R0 load a copy of row j mod R0 (unused): loads under a
        // branch would make the compiler wait for every load before the FFT
        const size_t off = zop_base(ky, kx0 / kTile, V.ntx, N, kTile) + min(kx0 + c, nxh - 1) +
                           (size_t)(act ? j : j % R0) * kTile;
        const QSM_GLOBAL float2* __restrict__ F = glb(V.spec[SPEC_A]) + off;
        const QSM_GLOBAL float* __restrict__ Q = glb(V.q) + off;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (HAS_F) fr[r] = ldg2<NT>(F + R0 * r * kTile);
            if constexpr (Q_MEM) qr[r] = Q[R0 * r * kTile];
        }
    }
    tws.commit(twl);
    // the multiplier's per-plane terms, once per block for every column
    __shared__ float4 zqt[Q_MEM ? 1 : N];
    if constexpr (!Q_MEM) {
        for (int kz = threadIdx.x; kz < N; kz += kThreads) zqt[kz] = TvQ::plane(V, kz, N);
    }
    C::template a_fwd<false>(threadIdx.x, v, lds);
    __syncthreads();
    if constexpr (!Q_MEM) {
        // the tile is in LDS and the operands are in flight: form q here
        TvQ tq;
        int fx, fy;
        pk_freq(V, min(kx0 + c, nxh - 1), ky, fx, fy);
        tq.init(V, fx, fy);
        if (act) {
            float4 pz[16];  // all LDS reads issued before the first use
#pragma unroll
            for (int r = 0; r < 16; ++r) pz[r] = zqt[j + R0 * r];
#pragma unroll
            for (int r = 0; r < 16; ++r) qr[r] = tq.at_plane(j + R0 * r, N, pz[r]);
        }
    }
    C::template b_fwd<false>(threadIdx.x, v, lds, twl);
    // doubly packed column 0 (block-uniform dpk): its entries go through LDS
    // so that each element can see Z(-kz); q at (0, ky) is qr, the Nyquist
    // plane's multiplier is formed here
    const bool dcol = dpk && c == 0 && act;
    if (dpk) {
        __syncthreads();  // every read of the first exchange is done
        if (dcol) {
#pragma unroll
            for (int r = 0; r < 16; ++r) lds[j + R0 * r] = v[r];
        }
        __syncthreads();
    }
    if (act) {
        TvQ tqB;
        if constexpr (!Q_MEM) {
            if (dcol) tqB.init(V, V.nx / 2, ky);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float2 qs = make_float2(qr[r] * v[r].x, qr[r] * v[r].y);
            if (dcol) {
                const int kz = j + R0 * r;
                float qB;
                if constexpr (Q_MEM) qB = glb(V.q)[q_nyq_base(V, ky) + kz];
                else qB = tqB.at_plane(kz, N, zqt[kz]);
                qs = pk_apply(v[r], lds[mirror_idx(kz, N)], qr[r], qB);
            }
            if constexpr (HAS_F)
                v[r] = make_float2(fr[r].x - qs.x, fr[r].y - qs.y);
            else
                v[r] = make_float2(-qs.x, -qs.y);
        }
    }
    __syncthreads();  // every read of the first exchange precedes the second's writes
    C::template lr_to_l16<true>(v, lds, twl);
    l16_store<R0>(v, buf, zs, kx0, nxh);
}

template <int N, int EG, int OP, int SCHED, int TW = kTile, bool NT = false>
__global__ __launch_bounds__(kThreads) void k_z_tv(const VolDesc* __restrict__ vols, LaunchTable lt,
                                                   const float2* __restrict__ tw,
                                                   const VolStatus* __restrict__ status) {
    constexpr int EMAX = col_emax(N, EG);
    constexpr bool TWO = SCHED == 0 && qsmfft::col2_ok(N) &&
                         (OP == ZOP_TV_SOLVE || OP == ZOP_TV_SOLVE0 || OP == ZOP_TV_ADJ || OP == ZOP_RTS_SOLVE);
    __shared__ float2 lds[TWO ? col_lds2(N, EG) : col_lds(N, EG)];
    __shared__ float2 twl[tw_lds(N, EG)];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    if (status && status[gv].done) return;
    static_assert(TW == kTile || N == 0, "compiled lengths use tiles of kTile columns");
    constexpr int L2 = tile_log2(TW);
    const int ntx = TW == kTile ? V.ntx : V.ntx_long;
    const int ky = lb / ntx;
    const int tx = lb - ky * ntx;
    const int kx0 = tx * TW;
    const int nxh = V.nxh;
    const int nz = N > 0 ? N : V.nz;
    const size_t zs = (size_t)nxh * V.ny;
    const size_t base = (size_t)ky * nxh;
    const int total = nz * TW;
    // f^ / q operands (tile-major): element (kx, kz) at fb + kx + kz * TW
    const size_t fb = zop_base(ky, tx, ntx, nz, TW);
    // column 0 holds two z spectra (the DC and Nyquist planes at ky = 0, ny/2)
    const bool dpk = pk_double(V, tx, ky);
    QSM_GLOBAL float2* buf = glb(V.spec[SPEC_WORK]) + base;
    TwStage<N, EG> tws;
    tws.fetch(tw, V.pz);
    if constexpr (TWO) {
        z_tv_col2<N, EG, OP, NT>(V, lds, twl, tws, ky, kx0, dpk);
        return;
    }
    if constexpr (OP == ZOP_TV_SOLVE0) {
        // g = 0 before the first step (AdmmBuffers::new), so div = 0 and x^ = f^
        col_load<EMAX, TW>(lds, glb(V.spec[SPEC_A]) + fb, TW, nz, kx0, nxh);
        tws.commit(twl);
        __syncthreads();
        run_fft<N, EG, EMAX, true, L2, true>(lds, V.pz, TW, TW, 1, twl, tw);
        col_store<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
        return;
    }
    col_load<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
    // FP64 multipliers: the z shares of L once per block, in flight of the
    // tile loads
    constexpr bool FP64_MULT = OP == ZOP_TV_SETUP || OP == ZOP_RTS_SETUP || OP == ZOP_TV_APPLYA ||
                               OP == ZOP_DIPOLE || OP == ZOP_FILTER;
    __shared__ double lzt[FP64_MULT && OP != ZOP_DIPOLE ? tw_lds(N, EG) : 1];
    const double* const lz = OP == ZOP_DIPOLE ? nullptr : lzt;
    SpecXY xy, xyB;
    if constexpr (FP64_MULT) {
        const int lap = lap_kind<OP>(V);
        if constexpr (OP != ZOP_DIPOLE)
            for (int kz = threadIdx.x; kz < nz; kz += kThreads) lzt[kz] = lap_axis(lap, kz, nz, V.vsz);
        int fx, fy;
        pk_freq(V, min(kx0 + (int)(threadIdx.x & (TW - 1)), nxh - 1), ky, fx, fy);
        xy.init(V, fx, fy, lap);
        if (dpk && (threadIdx.x & (TW - 1)) == 0) xyB.init(V, V.nx / 2, ky, lap);
    }
    // x-update operands, in flight during the forward FFT
    constexpr bool HAS_F = OP == ZOP_TV_SOLVE || OP == ZOP_RTS_SOLVE;
    constexpr bool Q_MEM = OP == ZOP_RTS_SOLVE;
    float2 fr[HAS_F ? EMAX : 1];
    float qr[Q_MEM ? EMAX : 1];
    if constexpr (HAS_F || Q_MEM) {
        const QSM_GLOBAL float2* __restrict__ F = glb(V.spec[SPEC_A]) + fb;
        const QSM_GLOBAL float* __restrict__ Q = glb(V.q) + fb;
#pragma unroll
        for (int t = 0; t < EMAX; ++t) {
            const int e = threadIdx.x + t * kThreads;
            const int kz = e >> L2;
            const int kx = kx0 + (e & (TW - 1));
            const bool in = e < total && kx < nxh;
            if constexpr (HAS_F) fr[t] = in ? ldg2<NT>(F + kx + kz * TW) : make_float2(0.0f, 0.0f);
            if constexpr (Q_MEM) qr[t] = in ? Q[kx + kz * TW] : 0.0f;
        }
    }
    tws.commit(twl);
    __syncthreads();
    run_fft<N, EG, EMAX, true, L2, false>(lds, V.pz, TW, TW, 1, twl, tw);
    // a thread's elements all lie in column c
    const int c = threadIdx.x & (TW - 1);
    const bool dcol = dpk && c == 0;
    // doubly packed column: Z(-kz) of each element, read before any is rewritten
    float2 zmir[EMAX];
    if (dpk) {
        if (dcol) {
#pragma unroll
            for (int t = 0; t < EMAX; ++t) {
                const int kz = min((int)(threadIdx.x + t * kThreads) >> L2, nz - 1);
                zmir[t] = lds[mirror_idx(kz, nz) * TW];
            }
        }
        __syncthreads();
    }
    if constexpr (OP == ZOP_TV_SETUP || OP == ZOP_RTS_SETUP) {
        QSM_GLOBAL float2* F = glb(V.spec[SPEC_A]) + fb;
        [[maybe_unused]] QSM_GLOBAL float* Q = glb(V.q) + fb;
#pragma unroll
        for (int t = 0; t < EMAX; ++t) {
            const int e = threadIdx.x + t * kThreads;
            const int kz = e >> L2;
            const int kx = kx0 + c;
            if (e < total && kx < nxh) {
                const float2 sv = lds[e];
                float2 fv;
                double m, qv;
                setup_mult<OP>(V, xy.at(kz, nz, lz), m, qv);
                if (dcol) {
                    double mB, qB;
                    setup_mult<OP>(V, xyB.at(kz, nz, lz), mB, qB);
                    fv = pk_apply_d(sv, zmir[t], m, mB);
                    if constexpr (OP == ZOP_RTS_SETUP) glb(V.q)[q_nyq_base(V, ky) + kz] = (float)qB;
                } else {
                    fv = make_float2((float)((double)sv.x * m), (float)((double)sv.y * m));
                }
                stg2(F + kx + kz * TW, fv);
                // (only RTS reads q back; TV forms it where it is used)
                if constexpr (OP == ZOP_RTS_SETUP) Q[kx + kz * TW] = (float)qv;
            }
        }
    } else {
        if constexpr (OP == ZOP_TV_APPLYA || OP == ZOP_DIPOLE || OP == ZOP_FILTER) {
#pragma unroll
            for (int t = 0; t < EMAX; ++t) {
                const int e = threadIdx.x + t * kThreads;
                const int kz = e >> L2;
                const int kx = kx0 + c;
                if (e < total) {
                    const float2 sv = lds[e];
                    float2 out = make_float2(0.0f, 0.0f);
                    if (kx < nxh) {
                        const double m = apply_mult<OP>(V, xy.at(kz, nz, lz));
                        if (dcol) {
                            out = pk_apply_d(sv, zmir[t], m, apply_mult<OP>(V, xyB.at(kz, nz, lz)));
                        } else {
                            out = make_float2((float)((double)sv.x * m), (float)((double)sv.y * m));
                        }
                    }
                    lds[e] = out;
                }
            }
        } else {
            TvQ tq, tqB;
            if constexpr (!Q_MEM) {
                int fx, fy;
                pk_freq(V, min(kx0 + c, nxh - 1), ky, fx, fy);
                tq.init(V, fx, fy);
                if (dcol) tqB.init(V, V.nx / 2, ky);
            }
#pragma unroll
            for (int t = 0; t < EMAX; ++t) {
                const int e = threadIdx.x + t * kThreads;
                if (e < total) {
                    const int kz = e >> L2;
                    const float2 sv = lds[e];
                    float2 qs;  // q * spectrum
                    if (dcol) {
                        float qA, qB;
                        if constexpr (Q_MEM) {
                            qA = qr[t];
                            qB = glb(V.q)[q_nyq_base(V, ky) + kz];
                        } else {
                            const float2 tz = ztw<N>(V, twl, kz, nz);
                            qA = tq.at(kz, nz, tz);
                            qB = tqB.at(kz, nz, tz);
                        }
                        qs = pk_apply(sv, zmir[t], qA, qB);
                    } else {
                        float q;
                        if constexpr (Q_MEM) q = qr[t];
                        else q = tq.at(kz, nz, ztw<N>(V, twl, kz, nz));
                        qs = make_float2(q * sv.x, q * sv.y);
                    }
                    if constexpr (HAS_F)
                        lds[e] = make_float2(fr[t].x - qs.x, fr[t].y - qs.y);
                    else
                        lds[e] = make_float2(-qs.x, -qs.y);
                }
            }
        }
        __syncthreads();
        run_fft<N, EG, EMAX, true, L2, true>(lds, V.pz, TW, TW, 1, twl, tw);
        col_store<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
    }
}

// ----------------------------------------------------------- C2R x passes --
// Rebuild the full complex row Z = A + iB from two half spectra (negative
// frequencies by conjugate symmetry; the imaginary parts of the DC and
// Nyquist bins are dropped, as Re(IFFT) of a full spectrum does).
// step 2: A, B = rows 2p, 2p+1 of sa; step 1: A = row p of sa, B = row p of sb.
template <int N, int EMAX>
__device__ __forceinline__ void c2r_load(float2* lds, const VolDesc& V, int nx, int nxh, int RB,
                                         const QSM_GLOBAL float2* __restrict__ sa,
                                         const QSM_GLOBAL float2* __restrict__ sb, int row0, int step,
                                         int nrows) {
    const int total = RB * nx;
    float2 r[EMAX];
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        const int p = div_nx<N>(e, V);
        const int k = e - p * nx;
        const bool neg = (2 * k > nx);
        const int kk = neg ? nx - k : k;
        // even nx: the Nyquist bin is the imaginary part of column 0
        const bool nyq = 2 * kk == nx;
        // rows past the volume (or past the block for e >= total) read its
        // last row: in bounds, and their outputs are never stored (each
        // half of the packed row is Hermitian, so they do not mix)
        const int ra = min(row0 + step * p, nrows - 1);
        const int rb = min((step == 2) ? row0 + step * p + 1 : row0 + step * p, nrows - 1);
        const int col = nyq ? 0 : kk;
        float2 A = ldg2(sa + col + (size_t)ra * nxh);
        float2 B = ldg2(sb + col + (size_t)rb * nxh);
        if (nyq) { A.x = A.y; B.x = B.y; }
        if (kk == 0 || nyq) { A.y = 0.0f; B.y = 0.0f; }
        if (neg) { A.y = -A.y; B.y = -B.y; }
        r[t] = make_float2(A.x - B.y, A.y + B.x);
    }
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < total) lds[e] = r[t];
    }
}

// c2r_load for compiled lengths divisible by 4: a thread takes two
// consecutive half-spectrum entries k0, k0 + 1 of a row pair (16-byte loads,
// every entry read once) and writes the full-spectrum elements they give:
// k and N - k for 0 < k < N / 2, and for k = 0 the DC element and the
// Nyquist element N / 2 (the imaginary parts of the packed column 0).
template <int N, int RB, bool NT>
__device__ __forceinline__ void c2r_load_pairs(float2* lds, const QSM_GLOBAL float2* __restrict__ sa,
                                               const QSM_GLOBAL float2* __restrict__ sb, int row0, int step,
                                               int nrows) {
    static_assert(N % 4 == 0, "pairs of half-spectrum entries");
    constexpr int NH = N / 2, NH2 = N / 4, TOT2 = RB * NH2;
    constexpr int T = (TOT2 + kThreads - 1) / kThreads;
    float4 a[T], b[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int e = threadIdx.x + t * kThreads;
        const int ec = e < TOT2 ? e : 0;  // idle threads load a valid pair (unused)
        const int p = ec / NH2;
        const int k0 = 2 * (ec - p * NH2);
        // rows past the volume read its last row: in bounds, never stored
        const int ra = min(row0 + step * p, nrows - 1);
        const int rb = min((step == 2) ? row0 + step * p + 1 : row0 + step * p, nrows - 1);
        a[t] = ldv<4, NT>((const QSM_GLOBAL float*)(sa + k0 + (size_t)ra * NH));
        b[t] = ldv<4, NT>((const QSM_GLOBAL float*)(sb + k0 + (size_t)rb * NH));
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < TOT2) {
            const int p = e / NH2;
            const int k0 = 2 * (e - p * NH2);
            float2* row = lds + p * N;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = k0 + c;
                const float2 A = c == 0 ? make_float2(a[t].x, a[t].y) : make_float2(a[t].z, a[t].w);
                const float2 B = c == 0 ? make_float2(b[t].x, b[t].y) : make_float2(b[t].z, b[t].w);
                if (k == 0) {
                    row[0] = make_float2(A.x, B.x);
                    row[NH] = make_float2(A.y, B.y);
                } else {
                    row[k] = make_float2(A.x - B.y, A.y + B.x);
                    row[N - k] = make_float2(A.x + B.y, B.x - A.y);
                }
            }
        }
    }
}

// c2r_load_pairs where it applies, else c2r_load.
template <int N, int RBC, int EMAX, bool NT = false>
__device__ __forceinline__ void c2r_load_rows(float2* lds, const VolDesc& V, int nx, int nxh, int RB,
                                              const QSM_GLOBAL float2* __restrict__ sa,
                                              const QSM_GLOBAL float2* __restrict__ sb, int row0, int step,
                                              int nrows) {
    if constexpr (N > 0 && N % 4 == 0) c2r_load_pairs<N, RBC, NT>(lds, sa, sb, row0, step, nrows);
    else c2r_load<N, EMAX>(lds, V, nx, nxh, RB, sa, sb, row0, step, nrows);
}

// TV: x_it = Re IFFT(x^) (src/inversion/admm.rs:111-114) and the two sums of
// relative_change (src/utils/mod.rs:69-77) accumulated in FP64 per block;
// the next pass's first block (or k_tv_reduce after the last iteration)
// reduces them.  no_change: nobody reads this iteration's sums (they are 0),
// so the previous iterate is not loaded; the pass is bound by memory, and 8
// bytes a voxel instead of 12 take 20.7 us instead of 25.1 at 256x256x160,
// 119 instead of 179 for two 384x384x256 volumes.
// MODE C2R_TV: as above.  C2R_ADJ: Re IFFT to adj_c (c-bar), nothing
// else.  C2R_F64: Re IFFT widened to f64 into adj_out.
// C2R_X0: FP32 into x[0], 0 where mask == 0 (src/utils/mask.rs:47-53; the RTS
// starting point, the closed-form inversions of host arrays).
enum C2RMode : int { C2R_TV = 0, C2R_ADJ = 1, C2R_F64 = 2, C2R_X0 = 3 };

template <int N, int EG, int MODE, int RBS = 0, bool NT = false>
__global__ __launch_bounds__(kThreads) void k_c2r_tv(const VolDesc* __restrict__ vols, LaunchTable lt,
                                                     const float2* __restrict__ tw, int parity,
                                                     const VolStatus* __restrict__ status, int no_change) {
    // half the R2C pass's pair-rows (after its row shift RBS), at least 1
    constexpr int RBF = N > 0 ? ((qsmfft::fixed_rows(N) >> RBS) / 2 > 0 ? (qsmfft::fixed_rows(N) >> RBS) / 2 : 1) : 0;
    constexpr int EMAX = N > 0 ? (RBF * N + kThreads - 1) / kThreads : kRowEmaxRt;
    __shared__ float2 lds[N > 0 ? RBF * N : kThreads * kRowEmaxRt];
    __shared__ float2 twl[tw_lds(N, EG)];
    __shared__ double sh[kThreads / 64];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    if (status && status[gv].done) return;
    const int nx = N > 0 ? N : V.nx;
    const int nxh = (nx + 1) / 2;
    const int RB = N > 0 ? RBF : V.rows_c;
    const int nrows = V.ny * V.nz;
    const int row0 = lb * RB * 2;
    const int total = RB * nx;
    const QSM_GLOBAL float2* s = glb(V.spec[SPEC_WORK]);
    TwStage<N, EG> tws;
    tws.fetch(tw, V.px);
    c2r_load_rows<N, RBF, EMAX, NT>(lds, V, nx, nxh, RB, s, s, row0, 2, nrows);
    if constexpr (MODE != C2R_TV) {
        tws.commit(twl);
        __syncthreads();
        run_fft<N, EG, EMAX, false, 0, true, RBF>(lds, V.px, RB, 1, nx, twl, tw);
#pragma unroll
        for (int t = 0; t < EMAX; ++t) {
            const int e = threadIdx.x + t * kThreads;
            if (e < total) {
                const int p = div_nx<N>(e, V);
                const int i = e - p * nx;
                const int ra = row0 + 2 * p, rb = ra + 1;
                const float2 z = lds[e];
                if constexpr (MODE == C2R_ADJ) {
                    QSM_GLOBAL float* __restrict__ o = glb(V.adj_c);
                    if (ra < nrows) o[i + (size_t)ra * nx] = z.x;
                    if (rb < nrows) o[i + (size_t)rb * nx] = z.y;
                } else if constexpr (MODE == C2R_X0) {
                    const QSM_GLOBAL uint8_t* __restrict__ m = glb(V.mask);
                    QSM_GLOBAL float* __restrict__ o = glb(V.x[0]);
                    const size_t ia = i + (size_t)ra * nx, ib = i + (size_t)rb * nx;
                    if (ra < nrows) o[ia] = m[ia] ? z.x : 0.0f;
                    if (rb < nrows) o[ib] = m[ib] ? z.y : 0.0f;
                } else {
                    QSM_GLOBAL double* __restrict__ o = glb(V.adj_out);
                    if (ra < nrows) o[i + (size_t)ra * nx] = (double)z.x;
                    if (rb < nrows) o[i + (size_t)rb * nx] = (double)z.y;
                }
            }
        }
        return;
    }
    const QSM_GLOBAL float* __restrict__ xo = glb(V.x[parity]);
    QSM_GLOBAL float* __restrict__ xn = glb(V.x[parity ^ 1]);
    if constexpr (N > 0 && N % 4 == 0) {
        // four consecutive columns per thread: 16-byte loads of the previous
        // iterate and stores of the new one
        constexpr int E4 = (RBF * N / 4 + kThreads - 1) / kThreads;
        float4 xa[E4] = {}, xb[E4] = {};  // previous iterate, in flight during the inverse FFT
        if (!no_change) {
#pragma unroll
            for (int t = 0; t < E4; ++t) {
                const int e = 4 * (threadIdx.x + t * kThreads);
                const int p = e / N;
                const int i = e - p * N;
                // rows past the volume read its last row: always in bounds, never used
                const int ra = min(row0 + 2 * p, nrows - 1), rb = min(row0 + 2 * p + 1, nrows - 1);
                xa[t] = ldv<4>(xo + i + (size_t)ra * N);
                xb[t] = ldv<4>(xo + i + (size_t)rb * N);
            }
        }
        tws.commit(twl);
        __syncthreads();
        run_fft<N, EG, EMAX, false, 0, true, RBF>(lds, V.px, RB, 1, nx, twl, tw);
        double sd = 0.0, sx = 0.0;
        auto add = [&](const float* z, float4 prev) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const double d = (double)z[c] - (double)vel<4>(prev, c);
                sd += d * d;
                sx += (double)z[c] * (double)z[c];
            }
        };
#pragma unroll
        for (int t = 0; t < E4; ++t) {
            const int e = 4 * (threadIdx.x + t * kThreads);
            if (e < total) {
                const int p = e / N;
                const int i = e - p * N;
                const int ra = row0 + 2 * p, rb = ra + 1;
                float za[4], zb[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float2 z = lds[e + c];
                    za[c] = z.x;
                    zb[c] = z.y;
                }
                if (ra < nrows) {
                    stv<4>(xn + i + (size_t)ra * N, vpack<4>(za));
                    if (!no_change) add(za, xa[t]);
                }
                if (rb < nrows) {
                    stv<4>(xn + i + (size_t)rb * N, vpack<4>(zb));
                    if (!no_change) add(zb, xb[t]);
                }
            }
        }
        const double tsd = block_sum(sd, sh);
        const double tsx = block_sum(sx, sh);
        if (threadIdx.x == 0) {
            QSM_GLOBAL double* part = glb(V.partial);
            part[2 * lb] = tsd;
            part[2 * lb + 1] = tsx;
        }
        return;
    }
    float2 xp[EMAX] = {};  // previous iterate, in flight during the inverse FFT
    if (!no_change) {
#pragma unroll
        for (int t = 0; t < EMAX; ++t) {
            const int e = threadIdx.x + t * kThreads;
            const int p = div_nx<N>(e, V);
            const int i = e - p * nx;
            // rows past the volume read its last row: always in bounds, never used
            const int ra = min(row0 + 2 * p, nrows - 1), rb = min(row0 + 2 * p + 1, nrows - 1);
            xp[t].x = xo[i + (size_t)ra * nx];
            xp[t].y = xo[i + (size_t)rb * nx];
        }
    }
    tws.commit(twl);
    __syncthreads();
    run_fft<N, EG, EMAX, false, 0, true, RBF>(lds, V.px, RB, 1, nx, twl, tw);
    double sd = 0.0, sx = 0.0;
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < total) {
            const int p = div_nx<N>(e, V);
            const int i = e - p * nx;
            const int ra = row0 + 2 * p, rb = ra + 1;
            const float2 z = lds[e];
            if (ra < nrows) {
                const double d = (double)z.x - (double)xp[t].x;
                xn[i + (size_t)ra * nx] = z.x;
                if (!no_change) {
                    sd += d * d;
                    sx += (double)z.x * (double)z.x;
                }
            }
            if (rb < nrows) {
                const double d = (double)z.y - (double)xp[t].y;
                xn[i + (size_t)rb * nx] = z.y;
                if (!no_change) {
                    sd += d * d;
                    sx += (double)z.y * (double)z.y;
                }
            }
        }
    }
    const double tsd = block_sum(sd, sh);
    const double tsx = block_sum(sx, sh);
    if (threadIdx.x == 0) {
        QSM_GLOBAL double* part = glb(V.partial);
        part[2 * lb] = tsd;
        part[2 * lb + 1] = tsx;
    }
}

// ------------------------------------------------ V-SHARP spectral passes --
// VS_FWD: forward z only (finishes FFT(field) / FFT(mask) in spec[sel]).
// VS_RADIUS: SPEC_WORK holds the x/y-transformed sphere indicator; forward z
//   gives S^ = Re / count (the normalised kernel, src/kernels/smv.rs:57-64);
//   P = M^ S^ / N -> SPEC_WORK and Q = F^ (1 - S^) / N -> SPEC_C, each
//   inverse-transformed along z (SPEC_A = F^, SPEC_B = M^).  The first
//   (largest) radius also keeps S^ for the deconvolution
//   (src/bgremove/vsharp.rs:147-156).
// VS_DECONV: forward z of FFT(local), X / (1 - S^) with |1 - S^| < threshold
//   -> 0 (src/bgremove/vsharp.rs:180-196; division form of
//   src/bgremove/sharp.rs:113-123 when divide != 0), scaled by 1/N, inverse z.
template <int N, int EG, int OP, int TW = kTile>
__global__ __launch_bounds__(kThreads) void k_z_vs(const VolDesc* __restrict__ vols, LaunchTable lt,
                                                   const float2* __restrict__ tw, int sel, int ridx,
                                                   int flag) {
    constexpr int EMAX = col_emax(N, EG);
    __shared__ float2 lds[col_lds(N, EG)];
    __shared__ float2 twl[tw_lds(N, EG)];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    static_assert(TW == kTile || N == 0, "compiled lengths use tiles of kTile columns");
    constexpr int L2 = tile_log2(TW);
    const int ntx = TW == kTile ? V.ntx : V.ntx_long;
    const int ky = lb / ntx;
    const int tx = lb - ky * ntx;
    const int kx0 = tx * TW;
    const int nxh = V.nxh;
    const int nz = N > 0 ? N : V.nz;
    const size_t zs = (size_t)nxh * V.ny;
    const size_t base = (size_t)ky * nxh;
    const int total = nz * TW;
    QSM_GLOBAL float2* buf = glb(V.spec[OP == ZOP_VS_FWD ? sel : SPEC_WORK]) + base;
    TwStage<N, EG> tws;
    tws.fetch(tw, V.pz);
    col_load<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
    tws.commit(twl);
    __syncthreads();
    run_fft<N, EG, EMAX, true, L2, false>(lds, V.pz, TW, TW, 1, twl, tw);
    if constexpr (OP == ZOP_VS_FWD) {
        col_store<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
    } else {
        // column 0 of tile 0 at ky = 0, ny/2 holds two z spectra (the DC and
        // Nyquist planes, even nx); the sphere's spectrum there is SA + i SB,
        // both real, and the S^ of the Nyquist plane is kept after the half
        // spectrum in vs_sfirst (2 nz entries)
        const bool dpk = pk_double(V, tx, ky);
        const int c = threadIdx.x & (TW - 1);
        const bool dcol = dpk && c == 0;
        QSM_GLOBAL float* sfirst = glb(V.vs_sfirst) + base;
        QSM_GLOBAL float* sfirst_nyq =
            glb(V.vs_sfirst) + (size_t)nxh * V.ny * V.nz + (ky == 0 ? 0 : (size_t)nz);
        if constexpr (OP == ZOP_VS_RADIUS) {
            const float inv_count = (float)(1.0 / V.vs_counts[ridx]);
            const float invN = (float)(1.0 / ((double)V.nx * V.ny * V.nz));
            const QSM_GLOBAL float2* __restrict__ FH = glb(V.spec[SPEC_A]) + base;
            const QSM_GLOBAL float2* __restrict__ MH = glb(V.spec[SPEC_B]) + base;
            float2 qv[EMAX];  // F^ (1 - S^) / N, transformed after P
#pragma unroll
            for (int t = 0; t < EMAX; ++t) {
                const int e = threadIdx.x + t * kThreads;
                if (e < total) {
                    const int kz = e >> L2;
                    const int kx = kx0 + c;
                    const float2 z = lds[e];
                    if (kx < nxh) {
                        const float2 m = ldg2(MH + kx + kz * zs);
                        const float2 fh = ldg2(FH + kx + kz * zs);
                        if (dcol) {
                            const int mz = mirror_idx(kz, nz);
                            const float sA = z.x * inv_count, sB = z.y * inv_count;
                            if (flag) {
                                sfirst[kx + kz * zs] = sA;
                                sfirst_nyq[kz] = sB;
                            }
                            const float2 mm = ldg2(MH + kx + mz * zs), fm = ldg2(FH + kx + mz * zs);
                            lds[e] = pk_apply(m, mm, sA * invN, sB * invN);
                            qv[t] = pk_apply(fh, fm, (1.0f - sA) * invN, (1.0f - sB) * invN);
                        } else {
                            const float sv = z.x * inv_count;
                            if (flag) sfirst[kx + kz * zs] = sv;
                            lds[e] = make_float2(m.x * sv * invN, m.y * sv * invN);
                            const float hp = (1.0f - sv) * invN;
                            qv[t] = make_float2(fh.x * hp, fh.y * hp);
                        }
                    } else {
                        lds[e] = make_float2(0.0f, 0.0f);
                        qv[t] = make_float2(0.0f, 0.0f);
                    }
                }
            }
            __syncthreads();
            run_fft<N, EG, EMAX, true, L2, true>(lds, V.pz, TW, TW, 1, twl, tw);
            col_store<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
            __syncthreads();
#pragma unroll
            for (int t = 0; t < EMAX; ++t) {
                const int e = threadIdx.x + t * kThreads;
                if (e < total) lds[e] = qv[t];
            }
            __syncthreads();
            run_fft<N, EG, EMAX, true, L2, true>(lds, V.pz, TW, TW, 1, twl, tw);
            col_store<EMAX, TW>(lds, glb(V.spec[SPEC_C]) + base, zs, nz, kx0, nxh);
        } else {  // ZOP_VS_DECONV
            const double invN = 1.0 / ((double)V.nx * V.ny * V.nz);
            // X / (1 - S^), 0 where |1 - S^| < threshold
            auto deconv = [&](double oms) {
                if (fabs(oms) < V.vs_threshold) return 0.0;
                return flag ? invN / oms : (1.0 / oms) * invN;
            };
            float2 zmir[EMAX];
            if (dpk) {
                if (dcol) {
#pragma unroll
                    for (int t = 0; t < EMAX; ++t) {
                        const int kz = min((int)(threadIdx.x + t * kThreads) >> L2, nz - 1);
                        zmir[t] = lds[mirror_idx(kz, nz) * TW];
                    }
                }
                __syncthreads();
            }
#pragma unroll
            for (int t = 0; t < EMAX; ++t) {
                const int e = threadIdx.x + t * kThreads;
                const int kz = e >> L2;
                const int kx = kx0 + c;
                if (e < total && kx < nxh) {
                    const float2 xv = lds[e];
                    const double oms = 1.0 - (double)sfirst[kx + kz * zs];
                    float2 y;
                    if (dcol) {
                        y = pk_apply_d(xv, zmir[t], deconv(oms), deconv(1.0 - (double)sfirst_nyq[kz]));
                    } else {
                        const double sc = deconv(oms);
                        y = make_float2((float)(xv.x * sc), (float)(xv.y * sc));
                    }
                    lds[e] = y;
                }
            }
            __syncthreads();
            run_fft<N, EG, EMAX, true, L2, true>(lds, V.pz, TW, TW, 1, twl, tw);
            col_store<EMAX, TW>(lds, buf, zs, nz, kx0, nxh);
        }
    }
}

// Row pass of one radius: Z = P + iQ per row, one inverse FFT; Re = mask
// convolution (src/kernels/smv.rs:79-105), Im = high-passed field
// (src/bgremove/vsharp.rs:163-168).  Erosion keeps a voxel when
// conv > delta; conv times the sphere's voxel count is an integer
// neighbour count, so it is rounded and the test is made on that integer in
// FP64, which reproduces the reference's f64 decision.  A voxel takes the
// value of the first (largest) radius whose eroded mask contains it
// (src/bgremove/vsharp.rs:170-176).
template <int N, int EG>
__global__ __launch_bounds__(kThreads) void k_c2r_vs_select(const VolDesc* __restrict__ vols,
                                                            LaunchTable lt,
                                                            const float2* __restrict__ tw, int ridx,
                                                            double delta) {
    constexpr int EMAX = x_emax(N, EG);
    __shared__ float2 lds[x_lds(N, EG)];
    __shared__ float2 twl[tw_lds(N, EG)];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    const int nx = N > 0 ? N : V.nx;
    const int nxh = (nx + 1) / 2;
    const int RB = N > 0 ? qsmfft::fixed_rows(N) : V.rows_x;
    const int nrows = V.ny * V.nz;
    const int row0 = lb * RB;
    TwStage<N, EG> tws;
    tws.fetch(tw, V.px);
    c2r_load_rows<N, (N > 0 ? qsmfft::fixed_rows(N) : 0), EMAX>(lds, V, nx, nxh, RB, glb(V.spec[SPEC_WORK]),
                                                            glb(V.spec[SPEC_C]), row0, 1, nrows);
    tws.commit(twl);
    QSM_GLOBAL uint8_t* fin = glb(V.vs_final);
    QSM_GLOBAL float* loc = glb(V.vs_local);
    __syncthreads();
    run_fft<N, EG, EMAX, false, 0, true>(lds, V.px, RB, 1, nx, twl, tw);
    const double count = V.vs_counts[ridx];
    const float countf = (float)count;
    const double norm = 1.0 / count;
    const int total = RB * nx;
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        const int p = div_nx<N>(e, V);
        const int i = e - p * nx;
        const int r = row0 + p;
        if (e < total && r < nrows) {
            const size_t idx = i + (size_t)r * nx;
            const float2 z = lds[e];
            const float k = rintf(z.x * countf);
            if ((double)k * norm > delta && !fin[idx]) {
                loc[idx] = z.y;
                fin[idx] = 1;
            }
        }
    }
}

// Final rows: local = Re IFFT(.) inside the final mask, 0 outside
// (src/bgremove/vsharp.rs:194-196); also writes the 0/1 mask.
template <int N, int EG>
__global__ __launch_bounds__(kThreads) void k_c2r_vs_out(const VolDesc* __restrict__ vols, LaunchTable lt,
                                                         const float2* __restrict__ tw) {
    constexpr int EMAX = x_emax(N, EG);
    __shared__ float2 lds[x_lds(N, EG)];
    __shared__ float2 twl[tw_lds(N, EG)];
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    int lb;
    const int gv = locate(lt, bid, lb);
    const VolDesc& V = vols[gv];
    const int nx = N > 0 ? N : V.nx;
    const int nxh = (nx + 1) / 2;
    const int RB = N > 0 ? qsmfft::fixed_rows(N) : V.rows_x;
    const int nrows = V.ny * V.nz;
    const int row0 = lb * RB * 2;
    const QSM_GLOBAL float2* s = glb(V.spec[SPEC_WORK]);
    TwStage<N, EG> tws;
    tws.fetch(tw, V.px);
    c2r_load_rows<N, (N > 0 ? qsmfft::fixed_rows(N) : 0), EMAX>(lds, V, nx, nxh, RB, s, s, row0, 2, nrows);
    tws.commit(twl);
    __syncthreads();
    run_fft<N, EG, EMAX, false, 0, true>(lds, V.px, RB, 1, nx, twl, tw);
    const int total = RB * nx;
    const QSM_GLOBAL uint8_t* fin = glb(V.vs_final);
    QSM_GLOBAL double* out = glb(V.out);
    QSM_GLOBAL float* out32 = glb(V.out32);
    auto put = [&](size_t idx, float v) {
        if (V.out32) out32[idx] = v;
        else out[idx] = (double)v;
    };
    QSM_GLOBAL uint8_t* mout = glb(V.mask_out);
#pragma unroll
    for (int t = 0; t < EMAX; ++t) {
        const int e = threadIdx.x + t * kThreads;
        if (e < total) {
            const int p = div_nx<N>(e, V);
            const int i = e - p * nx;
            const int ra = row0 + 2 * p, rb = ra + 1;
            const float2 z = lds[e];
            if (ra < nrows) {
                const size_t idx = i + (size_t)ra * nx;
                const uint8_t fm = fin[idx];
                put(idx, fm == 1 ? z.x : 0.0f);
                mout[idx] = fm;
            }
            if (rb < nrows) {
                const size_t idx = i + (size_t)rb * nx;
                const uint8_t fm = fin[idx];
                put(idx, fm == 1 ? z.y : 0.0f);
                mout[idx] = fm;
            }
        }
    }
}

}  // namespace qsm
