// Host runtime of the gfx950 QSM library: planning, device workspaces, the
// iteration loop with the reference's progress semantics, and the extern "C"
// entry points declared in include/qsm_gpu.h.
#include "qsm_internal.hpp"
#include "fft_dense.hpp"
#include "fft_chirp.hpp"
#include "qsm_hostmem.hpp"
#include "../../include/qsm_gpu.h"

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <atomic>
#include <map>
#include <numeric>
#include <mutex>
#include <string>
#include <vector>

namespace qsm {

void launch_tv_output(hipStream_t st, const VolDesc* d, const LaunchTable& lt, const VolStatus* status);
void launch_fill_zero(hipStream_t st, float* p, size_t n);
void launch_status_reset(hipStream_t st, VolStatus* s, int nvol);
void launch_vs_init(hipStream_t st, const VolDesc* d, const LaunchTable& lt);
void launch_tv_lbar(hipStream_t st, const VolDesc* d, int nvol, int nrows);
void launch_nltv_weights(hipStream_t st, const VolDesc* d, const LaunchTable& lt, int parity, int sel);
void launch_nltv_wmax(hipStream_t st, const VolDesc* d, int nvol, int nblk, int sel);
void launch_nltv_init(hipStream_t st, const VolDesc* d, const LaunchTable& lt);
void launch_status_clear_done(hipStream_t st, VolStatus* s, int nvol);
void launch_copy_probe(hipStream_t st, const float2* a, float2* b, size_t n);
int launch_stream_probe(hipStream_t st, int reads, int writes, const float* in, float* out, size_t n);
bool fixed_length(int n);

// ------------------------------------------------------------ error state --
thread_local std::string g_err;

int fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define QSM_HIP(call)                                                                  \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess)                                                          \
            return fail(e_ == hipErrorOutOfMemory ? QSM_ENOMEM : QSM_EHIP, "%s: %s (%s:%d)", \
                        #call, hipGetErrorString(e_), __FILE__, __LINE__);            \
    } while (0)

#define QSM_CHECK_LAUNCH()                                                             \
    do {                                                                               \
        hipError_t e_ = hipGetLastError();                                             \
        if (e_ != hipSuccess)                                                          \
            return fail(QSM_EHIP, "kernel launch: %s (%s:%d)", hipGetErrorString(e_),  \
                        __FILE__, __LINE__);                                           \
    } while (0)

// -------------------------------------------------------------- planning --
constexpr int kMaxLen = qsmfft::kMaxDirectLen;
using qsmfft::direct_length;
using qsmfft::chirp_length;
using qsmfft::chirp_tables;
using qsmfft::kMaxChirpLen;
bool length_ok(size_t n) {
    if (n < 1 || n > (size_t)kMaxLen) return false;
    return direct_length((int)n) || ((int)n <= kMaxChirpLen && chirp_length((int)n) > 0);
}

bool dense_length(int n) {
    int r[3], st;
    return !has_fixed_kernels(n) && qsmfft::dense_factorize(n, r, &st);
}

// Length the FFT stages of an axis of length n run at (n, or the chirp-z
// convolution length), which sizes the LDS tiles.
int work_length(int n) { return dense_length(n) || direct_length(n) ? n : chirp_length(n); }

// Dense column lengths up to 256 that take half tiles (kTileLong columns, 8
// elements per thread): a z pass keeps 3 waves per SIMD instead of 2 (80 -> 62
// us at 205, 82 -> 67 at 231), a y pass gains up to a tenth (27 -> 25 us at 250).
// Not where a dense radix has fewer than 4 butterflies a column (8 columns then
// fill half of a 16-wide matrix tile: the y pass at 211 29 -> 38 us), nor below
// 128 rows (too little work per block: z at 66 13.6 -> 16.2 us).
static bool half_tile(int n) {
    int r[qsmfft::kMaxStages], st = 0;
    if (n < 128 || n > 256 || !qsmfft::dense_factorize(n, r, &st)) return false;
    for (int s = 0; s < st; ++s)
        if (r[s] > qsmfft::kMaxRegRadix && n / r[s] < 4) return false;
    return true;
}

// Columns per tile of a column pass of length n: kTile up to 256 and for the
// compiled lengths, kTileLong above (a tile of 4096 elements at most, so four
// blocks fit a CU's LDS) and in half tiles.
int col_tile(int n) {
    if (has_fixed_kernels(n)) return kTile;
    return work_length(n) > 256 || half_tile(n) ? kTileLong : kTile;
}

// Launch size of a pass of length n (compiled kernels ignore it): the EG of
// the kernels that serve it, plus kColLongTile for dense column kernels above
// 256, in tiles of kTileLong columns.
int emax_for(int n, bool column) {
    if (dense_length(n)) {
        if (column && n > 256) return kEgDense + 16 + kColLongTile;
        return kEgDense + (column && col_tile(n) == kTileLong ? 8 : 16);
    }
    return column ? 32 : 16;
}

// Elements of the tile-major TV / RTS z-pass operands (f^, q) of a volume:
// ny * nz rows of whole z-pass tiles (at least the half spectrum).
size_t zop_elems(const VolDesc& V) {
    const int tw = col_tile(V.nz);
    const size_t cols = (size_t)(tw == kTile ? V.ntx : V.ntx_long) * tw;
    return cols * V.ny * V.nz;
}

// exp(-2 pi i q/n) from an exactly reduced angle, rounded once
inline float2 twiddle_entry(int q, int n) {
    long double a = -2.0L * 3.14159265358979323846264338327950288L * q / n;
    return make_float2((float)cosl(a), (float)sinl(a));
}

// The FFT tables of a length, formed in long double once per process (60 us
// for a 192x192x128 volume, 10 ms for a chirp-z filter of 1024) and kept:
// there are at most kMaxLen lengths, and kMaxDenseRadix dense radices.
// Kinds: 0 the twiddles of length n, 1 a dense radix's coefficients, 2 the
// chirp of length n and then its filter.
const std::vector<float2>& fft_table(int kind, int n) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::vector<float2>> tab;
    std::lock_guard<std::mutex> lk(mu);
    auto it = tab.find({kind, n});
    if (it != tab.end()) return it->second;
    // formed whole before it is kept: a host allocation may fail on the way
    std::vector<float2> t;
    if (kind == 0) {
        t.reserve(n);
        for (int q = 0; q < n; ++q) t.push_back(twiddle_entry(q, n));
    } else if (kind == 1) {
        t.resize(qsmfft::dense_table_len(n));
        qsmfft::dense_table(n, t.data());
    } else {
        std::vector<float2> f;
        chirp_tables(n, chirp_length(n), t, f);
        t.insert(t.end(), f.begin(), f.end());
    }
    return tab.emplace(std::make_pair(kind, n), std::move(t)).first->second;  // (stays valid as the map grows)
}

// The tables of the lengths of a set of volumes, end to end.
struct TwiddleBank {
    std::vector<float2> host;
    std::map<std::pair<int, int>, int> off;
    int put(int kind, int n) {
        auto it = off.find({kind, n});
        if (it != off.end()) return it->second;
        const int o = (int)host.size();
        const std::vector<float2>& t = fft_table(kind, n);
        host.insert(host.end(), t.begin(), t.end());
        off[{kind, n}] = o;
        return o;
    }
    int add(int n) { return put(0, n); }
    int add_dense(int R) { return put(1, R); }
    // chirp (n entries) and filter (M entries) offsets of length n
    void add_chirp(int n, int& oc, int& of) {
        oc = put(2, n);
        of = oc + n;
    }
};

qsmfft::Plan make_plan(int n, TwiddleBank& tb) {
    qsmfft::Plan p{};
    if (dense_length(n)) {
        qsmfft::make_dense_plan(n, p);
        p.tw_off = tb.add(n);
        for (int s = 0; s < p.nstages; ++s)
            if (p.radix[s] > qsmfft::kMaxRegRadix) p.dn_off[s] = tb.add_dense(p.radix[s]);
        return p;
    }
    if (direct_length(n)) {
        qsmfft::make_plan_stages(n, p);
        p.tw_off = tb.add(n);
        return p;
    }
    // chirp-z: the stages run at the convolution length
    const int M = chirp_length(n);
    qsmfft::make_plan_stages(M, p);
    p.tw_off = tb.add(M);
    p.bl_n = n;
    tb.add_chirp(n, p.bl_chirp, p.bl_filt);
    return p;
}

template <class T>
int dev_alloc(T** p, size_t count) {
    if (count == 0) count = 1;
    hipError_t e = workspace_alloc((void**)p, count * sizeof(T));
    if (e != hipSuccess)
        return fail(e == hipErrorOutOfMemory ? QSM_ENOMEM : QSM_EHIP, "hipMalloc(%zu bytes): %s",
                    count * sizeof(T), hipGetErrorString(e));
    return QSM_OK;
}

// Volume descriptors and FFT tables in one block, uploaded by one copy on the
// null stream (which, as ever, waits for work the caller left there).
int upload_plan(const VolDesc* vols, size_t n_vols, const TwiddleBank& tb, void** block, VolDesc** d_vols,
                float2** d_tw) {
    const size_t head = (n_vols * sizeof(VolDesc) + 255) / 256 * 256, tw = tb.host.size() * sizeof(float2);
    std::vector<unsigned char> host(head + tw);
    std::memcpy(host.data(), vols, n_vols * sizeof(VolDesc));
    if (tw) std::memcpy(host.data() + head, tb.host.data(), tw);
    unsigned char* d = nullptr;
    const int rc = dev_alloc(&d, host.size());
    if (rc) return rc;
    *block = d;
    *d_vols = reinterpret_cast<VolDesc*>(d);
    *d_tw = reinterpret_cast<float2*>(d + head);
    const hipError_t e = hipMemcpy(d, host.data(), host.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) return fail(QSM_EHIP, "hipMemcpy of plan tables: %s", hipGetErrorString(e));
    return QSM_OK;
}

int validate_grid(const qsm_grid* g) {
    if (!g) return fail(QSM_EPARAM, "grid is null");
    if (g->nx == 0 || g->ny == 0 || g->nz == 0) return fail(QSM_EPARAM, "grid has a zero dimension");
    if (!(g->vsx > 0) || !(g->vsy > 0) || !(g->vsz > 0))
        return fail(QSM_EPARAM, "voxel sizes must be positive");
    const size_t dims[3] = {g->nx, g->ny, g->nz};
    for (size_t d : dims)
        if (!length_ok(d))
            return fail(QSM_EUNSUPPORTED,
                        "axis length %zu not supported by the GPU FFT (2^a3^b5^c7^d11^e13^f <= %d, "
                        "or any length <= %d)",
                        d, kMaxLen, kMaxChirpLen);
    if (g->nx * g->ny * g->nz > (size_t)1 << 29)
        return fail(QSM_EUNSUPPORTED, "volume of %zu voxels exceeds 2^29", g->nx * g->ny * g->nz);
    return QSM_OK;
}

// Fill the geometry part of a descriptor and the block counts of each pass.
struct PassBlocks {
    int xpass, cpass, ypass, zpass, out;
};

// Pair-rows per block of the x passes: as many as 16 elements per thread
// hold (kRowEmaxRt for the runtime-plan kernels), at most 32.
static int default_rows_x(int nx) {
    if (has_fixed_kernels(nx)) return qsmfft::fixed_rows(nx);
    const int tile = qsmfft::kThreads * (dense_length(nx) ? 16 : kRowEmaxRt);
    return std::max(1, std::min(32, tile / work_length(nx)));
}

// Rows per block (pair-rows, or rows of the V-SHARP selection) of the x passes
// of a dense length other than the TV C2R pass, for a launch over `rows` of
// them.  As few as fill the launch's rounds of resident blocks (kRowBlocks: 148
// registers leave three a CU): long blocks leave CUs idle, many short ones pay
// for their start.  R2C pass at 20 columns and 20160 pair-rows 18 us with 28
// rows, 20 with 32, 26 with 8; at 143 columns and 6912 pair-rows 22 us with 10
// rows, 29 with 28 or 6; at 338 and 1536, 18 us with 2, 27 with 12.  With a dense
// radix, where every CU still has a block, whole matrix tiles of 16 butterflies
// if others were padded by more than an eighth (R2C pass at 239 columns and 6912
// pair-rows: 40 us with 16 rows, 44 with 10, 69 with 4), else half a tile at
// least (251 and 1536: 25 us with 8, 31 with 2).
//
// ROWS_SINGLE: passes whose threads take single elements (all but the TV ones,
// whose fill works row by row): two for each thread at least (V-SHARP of
// 12x144x96: 177 us with 32 rows, 190 with 12); with a dense radix full blocks,
// which share the coefficients among most rows, where there are 1.5 for every CU
// (356x144x96: 593 us with 10 rows, 657 with 8; 398x64x48, 300 blocks: 457 with
// 10, 345 with 6).  ROWS_UNROLLED: `rows` are the volume's own, since the solver
// sums the threshold's gradient block by block, so six at least for batches (six
// volumes of 16x64x48, 10 iterations and their gradient: 0.87 ms with 6, 1.22
// with 2; one volume the same with both).
// The rows change no bit of any value.
constexpr size_t kCus = 256, kRowBlocks = 3 * kCus;
// The largest dense radix of a length in fft_dense.hpp's stages, 0: none.
static int dense_radix(int n) {
    int r[qsmfft::kMaxStages], st = 0;
    return qsmfft::dense_factorize(n, r, &st) && st && r[0] > qsmfft::kMaxRegRadix ? r[0] : 0;  // (the largest comes first)
}
enum RowUse { ROWS_TV, ROWS_UNROLLED, ROWS_SINGLE };
static int dense_rows_x(int n, size_t rows, RowUse use) {
    const bool single = use == ROWS_SINGLE;
    const size_t most = default_rows_x(n) & ~1, rounds = (rows + kRowBlocks * most - 1) / (kRowBlocks * most);
    const size_t least = single ? (2 * qsmfft::kThreads + n - 1) / n : (use == ROWS_UNROLLED ? 6 : 2);
    const auto even = [](size_t k) { return (k + 1) & ~(size_t)1; };  // the same rows for each of the fill's four waves
    size_t per = even(std::max((rows + kRowBlocks * rounds - 1) / (kRowBlocks * rounds), least));
    if (const int R = dense_radix(n)) {
        if (single && 2 * rows >= 3 * kCus * most) return (int)most;
        const size_t nb = n / R, whole = 16 / std::gcd((size_t)16, nb), used = nb * per;
        const size_t full = whole > most ? most
                                         : std::min(std::max(whole, (per + whole / 2) / whole * whole), most / whole * whole);
        if (rows < kCus * full) per = even(std::max(per, (8 + nb - 1) / nb));
        else if (9 * used < 8 * ((used + 15) / 16 * 16)) per = even(full);  // (padded by more than an eighth)
    }
    return (int)std::min(per, most);
}
static size_t pair_rows(const qsm_grid& g) { return (g.ny * g.nz + 1) / 2; }

// Pair-rows of the volumes of each x length, which share a launch.
template <class VOLS>
static std::map<size_t, size_t> length_pairs(const VOLS* vols, size_t n_vols) {
    std::map<size_t, size_t> pairs;
    for (size_t v = 0; v < n_vols; ++v) pairs[vols[v].grid.nx] += pair_rows(vols[v].grid);
    return pairs;
}

// rows, use: for dense lengths, see dense_rows_x.  xshift / cshift 2
// (compiled lengths): the R2C / TV C2R passes take a quarter of their default
// rows per block, as the kernels launched with PassArgs::xshift = 2 do (C2R:
// half the R2C pass's rows before its shift).
PassBlocks fill_geometry(VolDesc& V, const qsm_grid& g, TwiddleBank& tb, size_t rows, RowUse use,
                         int xshift = 0, int cshift = 0) {
    V.nx = (int)g.nx; V.ny = (int)g.ny; V.nz = (int)g.nz;
    V.nxh = (V.nx + 1) / 2;  // even nx: DC and Nyquist share column 0
    if (has_fixed_kernels(V.nx)) V.rows_x = qsmfft::shifted_rows(V.nx, xshift);
    else V.rows_x = dense_length(V.nx) ? dense_rows_x(V.nx, rows, use) : default_rows_x(V.nx);
    // compiled C2R kernels take half the R2C pass's pair-rows (the previous
    // iterate stays in registers across the transform), the others what their
    // tile of 8 elements per thread holds (fewer did not pay: 9 us with 12 to 32
    // rows, 16 with 4, at 20 columns and 6912 pair-rows), but with a dense radix
    // no more than leave every CU a block (82 columns, 1536 pair-rows: 10.9 us
    // with 4, 12.7 with 24).  The sums of the relative change follow these
    // blocks, so they depend on the volume's own shape only.
    if (has_fixed_kernels(V.nx)) {
        V.rows_c = std::max(1, (default_rows_x(V.nx) >> cshift) / 2);
    } else {
        V.rows_c = std::max(1, std::min(32, qsmfft::kThreads * kRowEmaxRt / work_length(V.nx)));
        if (dense_length(V.nx) && dense_radix(V.nx))
            V.rows_c = std::min(V.rows_c, (int)std::max<size_t>(4, (pair_rows(g) + kCus - 1) / kCus));
    }
    V.ntx = (V.nxh + kTile - 1) / kTile;
    V.ntx_long = (V.nxh + kTileLong - 1) / kTileLong;
    V.m_nx = qsmfft::magic_for((uint32_t)V.nx);
    V.m_nxh = qsmfft::magic_for((uint32_t)V.nxh);
    V.m_ny = qsmfft::magic_for((uint32_t)V.ny);
    V.px = make_plan(V.nx, tb);
    V.py = make_plan(V.ny, tb);
    V.pz = make_plan(V.nz, tb);
    V.vsx = g.vsx; V.vsy = g.vsy; V.vsz = g.vsz;
    V.hx = (float)(1.0 / g.vsx); V.hy = (float)(1.0 / g.vsy); V.hz = (float)(1.0 / g.vsz);
    PassBlocks pb;
    const int npairs = (int)pair_rows(g);
    pb.xpass = (npairs + V.rows_x - 1) / V.rows_x;
    pb.cpass = (npairs + V.rows_c - 1) / V.rows_c;
    pb.ypass = (col_tile(V.ny) == kTile ? V.ntx : V.ntx_long) * V.nz;
    pb.zpass = (col_tile(V.nz) == kTile ? V.ntx : V.ntx_long) * V.ny;
    const size_t N = (size_t)V.nx * V.ny * V.nz;
    pb.out = (int)((N + 1023) / 1024);
    return pb;
}

// Volumes of a batch grouped by the length of one pass axis: one launch per
// group, so each group runs the kernel compiled for its length.
struct PassGroup {
    int n;
    int emax;
    LaunchTable lt;
    int xshift = 0;  // x passes: row shift of every volume in the group
};
using Groups = std::vector<PassGroup>;

void launch_tv_reduce(hipStream_t st, const VolDesc* d, int nvol, VolStatus* status, VolStatus* mirror);

// shift (x passes): each volume's row shift; volumes of one length with
// different shifts run in separate groups.
Groups make_groups(const std::vector<int>& len, const std::vector<int>& blocks, bool column,
                   const std::vector<int>* shift = nullptr) {
    Groups gs;
    for (size_t v = 0; v < len.size(); ++v) {
        const int sh = shift ? (*shift)[v] : 0;
        PassGroup* g = nullptr;
        for (auto& x : gs)
            if (x.n == len[v] && x.xshift == sh) g = &x;
        if (!g) {
            gs.push_back(PassGroup{});
            g = &gs.back();
            g->n = len[v];
            g->emax = emax_for(len[v], column);
            g->xshift = sh;
            g->lt.nvol = 0;
            g->lt.start[0] = 0;
        }
        LaunchTable& lt = g->lt;
        lt.vol[lt.nvol] = (int)v;
        lt.start[lt.nvol + 1] = lt.start[lt.nvol] + blocks[v];
        ++lt.nvol;
    }
    return gs;
}

// ------------------------------------------------- column-pass schedules --
// Per (pass, axis length): 0 two-stage, 1 LDS-staged.  Pass 0: the y passes;
// pass 1: the per-iteration z passes.  Mode 0 (default): a fixed table, so
// every process computes the same bits; 1 always two-stage; 2 always staged;
// 3 tuned: the first batch using a length times both forms and the faster
// one is kept for the process (-1 in the table until then).
namespace {
constexpr int kMaxAxis = 512;
std::mutex g_sched_mu;
int8_t g_sched_tab[2][kMaxAxis + 1];
std::atomic<int> g_sched_mode{0};
struct SchedInit {
    SchedInit() { std::memset(g_sched_tab, -1, sizeof g_sched_tab); }
} g_sched_init;

int sched_pass(int kind) {
    if (kind == P_Y_FWD || kind == P_Y_INV) return 0;
    if (kind == P_Z_TV_SOLVE || kind == P_Z_TV_SOLVE0 || kind == P_Z_TV_ADJ || kind == P_Z_RTS_SOLVE) return 1;
    return -1;
}

// The fixed table: the forms the tuner chose on MI355X over the TV workloads
// (256x256x160, the uneven 32-volume batch): the staged form for y passes of
// length 144 and 176, where radices 9 and 11 in registers cost more than
// LDS stages, and the two-stage form everywhere else.
int fixed_schedule(int pass, int n) { return (pass == 0 && (n == 144 || n == 176)) ? 1 : 0; }
}  // namespace

int column_schedule(int kind, int n) {
    const int pass = sched_pass(kind);
    if (pass < 0 || n < 0 || n > kMaxAxis || !qsmfft::col2_ok(n)) return 1;
    const int mode = g_sched_mode.load();
    if (mode == 1) return 0;
    if (mode == 2) return 1;
    if (mode == 0) return fixed_schedule(pass, n);
    std::lock_guard<std::mutex> lk(g_sched_mu);
    const int t = g_sched_tab[pass][n];
    return t < 0 ? fixed_schedule(pass, n) : t;
}

void run_groups(int kind, const Groups& gs, const PassArgs& a) {
    PassArgs b = a;
    for (const auto& g : gs) {
        b.sched = column_schedule(kind, g.n);
        b.xshift = g.xshift;
        launch_pass(kind, g.n, g.emax, g.lt, b);
    }
}

LaunchTable identity_table(const std::vector<int>& blocks) {
    LaunchTable lt{};
    lt.nvol = (int)blocks.size();
    lt.start[0] = 0;
    for (size_t v = 0; v < blocks.size(); ++v) {
        lt.vol[v] = (int)v;
        lt.start[v + 1] = lt.start[v] + blocks[v];
    }
    return lt;
}

}  // namespace qsm

using namespace qsm;

// ============================================================ TV batch ====
struct qsm_tv_batch {
    int nvol = 0;
    int method = 0;  // 0 TV-ADMM (src/inversion/tv.rs), 1 RTS (src/inversion/rts.rs)
    // The fused z/u update clamps to [-t, t], t = lambda / rho >= 0; for any
    // other t (a negative lambda, say) the recording kernel, which forms
    // shrink itself, runs in its place with a scratch record, from the second
    // iteration on.
    bool plain_shrink = false;
    bool streams = false;  // larger than the Infinity Cache (kStreamBytes)
    bool field32 = false;  // the field is VolDesc::vs_local, in f32 (host entry points)
    void* host_out = nullptr;  // their result array, made ready while the device works
    size_t host_bytes = 0;
    qsm_tv_params params{};
    std::vector<VolDesc> h;
    VolDesc* d_vols = nullptr;
    VolStatus* d_status = nullptr;
    VolStatus* h_status = nullptr;   // pinned mirror written by the reduce kernel
    VolStatus* h_status_dev = nullptr;
    float2* d_tw = nullptr;
    Groups gx, gxc, gy, gz;         // x / TV C2R / y / z passes grouped by axis length
    LaunchTable lt_out{};
    std::vector<void*> allocs;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    static constexpr int kWindow = 4;
    PassArgs args(const VolStatus* status) const {
        PassArgs a{};
        a.stream = stream;
        a.vols = d_vols;
        a.tw = d_tw;
        a.status = status;
        a.status_rw = nullptr;
        a.mirror = nullptr;
        a.sel = SPEC_WORK;
        a.sel2 = -1;
        a.nt = streams ? 1 : 0;
        return a;
    }
    hipEvent_t ev[kWindow] = {};
    // Iterations it >= 2 replay captured graphs: graph p is one iteration with
    // (it - 1) & 1 == p (its kernel arguments depend only on the parity).
    // graph_state: 0 not built yet, 1 built, -1 eager launches (disabled, or
    // the stream cannot be captured).
    hipGraphExec_t gexec[2] = {};
    int graph_state = 0;
    // Passes with several launch groups (volumes of several axis lengths)
    // fork them over the batch's stream and up to kSide side streams and
    // join before the next pass, so the groups' last waves overlap.  Created
    // only for batches with more than one group in some pass.
    static constexpr int kSide = 3;
    hipStream_t side[kSide] = {};
    hipEvent_t ev_fork[5] = {};
    hipEvent_t ev_join[5][kSide] = {};
};

static void batch_free(qsm_tv_batch* b) {
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    for (auto& g : b->gexec)
        if (g) (void)hipGraphExecDestroy(g);
    for (auto& st : b->side)
        if (st) (void)hipStreamSynchronize(st);
    for (void* p : b->allocs) workspace_free(p);
    for (auto& e : b->ev_fork)
        if (e) (void)hipEventDestroy(e);
    for (auto& row : b->ev_join)
        for (auto& e : row)
            if (e) (void)hipEventDestroy(e);
    for (auto& st : b->side)
        stream_give(st);
    pinned_give(b->h_status);
    for (auto& e : b->ev)
        if (e) (void)hipEventDestroy(e);
    if (b->own_stream && b->stream) stream_give(b->stream);
    delete b;
}

// The autotuner (schedule mode 3): for every y and z length of a new batch
// that has no entry yet, time the forward y pass and the z solve pass under
// both schedules on the batch's own launch tables and buffers (before any
// run, so only scratch is overwritten, after clearing it so that no
// uninitialised values enter the timed launches; convergence flags are not
// consulted) and keep the faster one for the rest of the process.  One
// warm-up and the best of five timed launches each.  The two forms round
// differently, so tuned results can differ between processes in the last
// bits; the default mode uses the fixed table instead.
static int tune_column_schedules(qsm_tv_batch* B) {
    if (g_sched_mode.load() != 3) return QSM_OK;
    {
        // a stream under capture cannot be timed: keep the defaults
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(B->stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            return QSM_OK;
        }
    }
    for (const auto& V : B->h) {
        launch_fill_zero(B->stream, reinterpret_cast<float*>(V.spec[SPEC_WORK]), 2 * (size_t)V.nxh * V.ny * V.nz);
        launch_fill_zero(B->stream, reinterpret_cast<float*>(V.spec[SPEC_A]), 2 * zop_elems(V));
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    auto best_ms = [&](int kind, const PassGroup& g, int sched, float& best) {
        PassArgs a = B->args(nullptr);
        a.sched = sched;
        launch_pass(kind, g.n, g.emax, g.lt, a);
        best = 1e30f;
        for (int r = 0; r < 5 && e == hipSuccess; ++r) {
            float ms = 0.f;
            if ((e = hipEventRecord(e0, B->stream)) != hipSuccess) break;
            launch_pass(kind, g.n, g.emax, g.lt, a);
            if ((e = hipGetLastError()) != hipSuccess) break;
            if ((e = hipEventRecord(e1, B->stream)) != hipSuccess) break;
            if ((e = hipEventSynchronize(e1)) != hipSuccess) break;
            if ((e = hipEventElapsedTime(&ms, e0, e1)) != hipSuccess) break;
            best = std::min(best, ms);
        }
    };
    const struct { const Groups* gs; int kind; int pass; } work[2] = {
        {&B->gy, P_Y_FWD, 0}, {&B->gz, P_Z_TV_SOLVE, 1}};
    for (const auto& w : work) {
        for (const auto& g : *w.gs) {
            if (e != hipSuccess) break;
            if (g.n > kMaxAxis || !qsmfft::col2_ok(g.n)) continue;
            {
                std::lock_guard<std::mutex> lk(g_sched_mu);
                if (g_sched_tab[w.pass][g.n] >= 0) continue;
            }
            float t0 = 0.f, t1 = 0.f;
            best_ms(w.kind, g, 0, t0);
            best_ms(w.kind, g, 1, t1);
            if (e != hipSuccess) break;
            // the staged form only when clearly faster: measured at creation,
            // with the batch's data in cache, the two come closer than in the
            // iteration (where the two-stage y pass leads by ~9 % at 256)
            std::lock_guard<std::mutex> lk(g_sched_mu);
            g_sched_tab[w.pass][g.n] = (int8_t)(t1 < 0.97f * t0 ? 1 : 0);
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (e != hipSuccess) return fail(QSM_EHIP, "schedule tuning: %s", hipGetErrorString(e));
    return QSM_OK;
}

// rts != null selects RTS: its rho, tol, max_iter replace params' (params
// may then be null).
// io: the host entry points' one volume, whose field and output are f32 on the
// device (the volume's own d_field and d_chi are then null).  unrolled: the
// batch of an unrolled solver.
struct HostVolume {
    float* field = nullptr;
    float* chi = nullptr;
    uint8_t* mask = nullptr;
    double* out = nullptr;  // the caller's result array of n values
    size_t n = 0;
};
static int tv_batch_create_impl(const qsm_tv_volume* vols, size_t n_vols, const qsm_tv_params* params_in,
                                void* stream, qsm_tv_batch** out, const qsm_rts_params* rts = nullptr,
                                const HostVolume* io = nullptr, bool unrolled = false) {
    qsm_tv_params rts_as_tv{};
    if (rts) {
        if (!(rts->rho > 0) || std::isnan(rts->delta) || std::isnan(rts->mu))
            return fail(QSM_EPARAM, "RTS needs rho > 0 and finite delta, mu");
        rts_as_tv.lambda = 1.0;  // threshold 1/rho is set per volume below
        rts_as_tv.rho = rts->rho;
        rts_as_tv.tol = rts->tol;
        rts_as_tv.max_iter = rts->max_iter;
        params_in = &rts_as_tv;
    }
    const qsm_tv_params* params = params_in;
    if (!vols || !params || !out) return fail(QSM_EPARAM, "null argument");
    if (n_vols == 0 || n_vols > (size_t)kMaxVolumes)
        return fail(QSM_EPARAM, "batch size %zu outside 1..%d", n_vols, kMaxVolumes);
    if (!(params->rho != 0.0) || std::isnan(params->rho) || std::isnan(params->lambda))
        return fail(QSM_EPARAM, "rho must be non-zero and lambda/rho not NaN");
    for (size_t v = 0; v < n_vols; ++v) {
        int rc = validate_grid(&vols[v].grid);
        if (rc) return rc;
        if (!io && (!vols[v].d_field || !vols[v].d_mask || !vols[v].d_chi))
            return fail(QSM_EPARAM, "volume %zu has a null device pointer", v);
        const double* b = vols[v].bdir;
        double bn = std::sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
        if (!(bn > 0)) return fail(QSM_EPARAM, "volume %zu: B0 direction has zero length", v);
    }
    qsm_tv_batch* B = new qsm_tv_batch();
    B->nvol = (int)n_vols;
    B->method = rts ? 1 : 0;
    B->params = *params;
    B->h.resize(n_vols);
    TwiddleBank tb;
    std::vector<int> lx, ly, lz, bx, bc, by, bz, bo;
    auto cleanup = [&](int rc) { batch_free(B); return rc; };
    // A small volume of a compiled x length, whose R2C pass would launch
    // fewer than 1024 blocks (128 for 128x128x64 against ~768 resident), runs
    // that pass with a quarter of the rows per block, and its TV C2R pass
    // likewise, where either keeps at least 4 pair-rows per block (fewer made
    // the C2R pass slower, measured).  The choice depends on the volume's own
    // shape only: the two forms round differently in the last bits, and a
    // volume must give the same bits alone and in any batch.
    std::vector<int> xshift(n_vols), cshift(n_vols);
    for (size_t v = 0; v < n_vols; ++v) {
        const int nx = (int)vols[v].grid.nx, r0 = default_rows_x(nx), rc = std::max(1, r0 / 2);
        const long npairs = (long)pair_rows(vols[v].grid);
        const bool fixed = has_fixed_kernels(nx);
        xshift[v] = (fixed && (npairs + r0 - 1) / r0 < 1024 && (r0 >> 2) >= 4) ? 2 : 0;
        cshift[v] = (fixed && (npairs + rc - 1) / rc < 1024 && (r0 >> 2) / 2 >= 4) ? 2 : 0;
    }
    std::map<size_t, size_t> pairs = length_pairs(vols, n_vols);
    // (the quarter-row R2C pass has no non-temporal form: three 192x192x128
    // volumes, 566 MB, took 203 us an iteration, 205 with the other passes' forms)
    size_t voxels = 0;
    for (size_t v = 0; v < n_vols; ++v)
        if (!xshift[v]) voxels += vols[v].grid.nx * vols[v].grid.ny * vols[v].grid.nz;
    B->streams = voxels * kIterBytes > kStreamBytes;
    for (size_t v = 0; v < n_vols; ++v) {
        VolDesc& V = B->h[v];
        std::memset(&V, 0, sizeof V);
        const size_t rows = unrolled ? pair_rows(vols[v].grid) : pairs[vols[v].grid.nx];
        PassBlocks pb = fill_geometry(V, vols[v].grid, tb, rows, unrolled ? ROWS_UNROLLED : ROWS_TV, xshift[v], cshift[v]);
        const double* b = vols[v].bdir;
        double bn = std::sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
        V.bx = b[0] / bn; V.by = b[1] / bn; V.bz = b[2] / bn;  // src/kernels/dipole.rs:39-43
        V.rho = params->rho;
        V.tol = params->tol;
        V.thr = (float)(params->lambda / params->rho);          // src/inversion/tv.rs:78
        if (rts) {
            V.thr = (float)(1.0 / rts->rho);                     // src/inversion/rts.rs:191-201
            V.filt = 5;                                          // FILT_RTS_X0
            V.filt_a = rts->delta;
            V.filt_b = rts->mu;
            V.lsmr_iter = (int)rts->lsmr_iter;
        }
        if (!(V.thr >= 0.0f)) B->plain_shrink = true;
        V.field = vols[v].d_field;
        V.mask = vols[v].d_mask;
        V.out = vols[v].d_chi;
        if (io) {
            V.vs_local = io->field;
            V.mask = io->mask;
            V.out32 = io->chi;
            B->field32 = true;
        }
        lx.push_back(V.nx); bx.push_back(pb.xpass); bc.push_back(pb.cpass);
        ly.push_back(V.ny); by.push_back(pb.ypass);
        lz.push_back(V.nz); bz.push_back(pb.zpass);
        bo.push_back(pb.out);
        V.npartial = pb.cpass;
        const size_t N = (size_t)V.nx * V.ny * V.nz;
        const size_t Nh = (size_t)V.nxh * V.ny * V.nz;
        int rc;
        for (int p = 0; p < 2; ++p) {
            if ((rc = dev_alloc(&V.x[p], N + kRowSlack))) return cleanup(rc);
            B->allocs.push_back(V.x[p]);
            if ((rc = dev_alloc(&V.u[p], 3 * N + kRowSlack))) return cleanup(rc);
            B->allocs.push_back(V.u[p]);
        }
        if ((rc = dev_alloc(&V.spec[SPEC_WORK], Nh))) return cleanup(rc);
        B->allocs.push_back(V.spec[SPEC_WORK]);
        // f^ and q: tile-major z-pass operands (zop_base in the kernels)
        if ((rc = dev_alloc(&V.spec[SPEC_A], zop_elems(V)))) return cleanup(rc);
        B->allocs.push_back(V.spec[SPEC_A]);
        V.q_len = zop_elems(V);
        if (rts) {
            if ((rc = dev_alloc(&V.q, V.q_len + 2 * (size_t)V.nz))) return cleanup(rc);
            B->allocs.push_back(V.q);
        }
        if ((rc = dev_alloc(&V.partial, 2 * (size_t)pb.cpass))) return cleanup(rc);
        B->allocs.push_back(V.partial);
    }
    if (B->plain_shrink) {
        for (auto& V : B->h) {
            int rc;
            if ((rc = dev_alloc(&V.ckpt, 3 * (size_t)V.nx * V.ny * V.nz))) return cleanup(rc);
            B->allocs.push_back(V.ckpt);
        }
    }
    B->gx = make_groups(lx, bx, false, &xshift);
    B->gxc = make_groups(lx, bc, false, &cshift);
    B->gy = make_groups(ly, by, true);
    B->gz = make_groups(lz, bz, true);
    B->lt_out = identity_table(bo);
    int rc;
    if ((rc = dev_alloc(&B->d_status, n_vols))) return cleanup(rc);
    B->allocs.push_back(B->d_status);
    {
        static_assert(kMaxVolumes * sizeof(VolStatus) <= kPinnedBlock, "status mirror block");
        hipError_t e = pinned_take((void**)&B->h_status);
        if (e != hipSuccess) { B->h_status = nullptr; return cleanup(fail(QSM_EHIP, "hipHostMalloc: %s", hipGetErrorString(e))); }
        e = hipHostGetDevicePointer((void**)&B->h_status_dev, B->h_status, 0);
        if (e != hipSuccess) return cleanup(fail(QSM_EHIP, "hipHostGetDevicePointer: %s", hipGetErrorString(e)));
        std::memset(B->h_status, 0, n_vols * sizeof(VolStatus));
    }
    if (stream) {
        B->stream = (hipStream_t)stream;
    } else {
        hipError_t e = stream_take(&B->stream);
        if (e != hipSuccess) { B->stream = nullptr; return cleanup(fail(QSM_EHIP, "hipStreamCreate: %s", hipGetErrorString(e))); }
        B->own_stream = true;
    }
    for (auto& e : B->ev) {
        hipError_t he = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        if (he != hipSuccess) { e = nullptr; return cleanup(fail(QSM_EHIP, "hipEventCreate: %s", hipGetErrorString(he))); }
    }
    {
        void* block = nullptr;
        rc = upload_plan(B->h.data(), n_vols, tb, &block, &B->d_vols, &B->d_tw);
        if (block) B->allocs.push_back(block);
        if (rc) return cleanup(rc);
    }
    {
        int rc = tune_column_schedules(B);
        if (rc) return cleanup(rc);
    }
    if (B->gx.size() > 1 || B->gy.size() > 1 || B->gz.size() > 1 || B->gxc.size() > 1) {
        for (auto& st : B->side) {
            hipError_t e = stream_take(&st);
            if (e != hipSuccess) { st = nullptr; return cleanup(fail(QSM_EHIP, "hipStreamCreate: %s", hipGetErrorString(e))); }
        }
        auto mk = [&](hipEvent_t& ev) {
            hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
            if (e != hipSuccess) ev = nullptr;
            return e;
        };
        for (auto& ev : B->ev_fork)
            if (mk(ev) != hipSuccess) return cleanup(fail(QSM_EHIP, "hipEventCreate failed"));
        for (auto& row : B->ev_join)
            for (auto& ev : row)
                if (mk(ev) != hipSuccess) return cleanup(fail(QSM_EHIP, "hipEventCreate failed"));
    }
    *out = B;
    return QSM_OK;
}

// One TV-ADMM iteration (src/inversion/admm.rs:76-145) for every volume.
// Its first pass also closes iteration it-1 (relative change, convergence);
// `closed` (if set) is recorded right after that pass.
// One pass of an iteration over all groups: sequential on the batch's
// stream, or forked over the side streams (group i on lane i mod (S+1), lane
// 0 the batch's stream) and joined back.  slot: the pass's event set.
static int run_pass(qsm_tv_batch* B, int slot, int kind, const Groups& gs, const PassArgs& a) {
    if (gs.size() < 2 || !B->side[0]) {
        run_groups(kind, gs, a);
        return QSM_OK;
    }
    const int S = std::min<int>(qsm_tv_batch::kSide, (int)gs.size() - 1);
    QSM_HIP(hipEventRecord(B->ev_fork[slot], B->stream));
    for (int s = 0; s < S; ++s) QSM_HIP(hipStreamWaitEvent(B->side[s], B->ev_fork[slot], 0));
    PassArgs b = a;
    for (size_t i = 0; i < gs.size(); ++i) {
        const int lane = (int)(i % (size_t)(S + 1));
        b.stream = lane == 0 ? B->stream : B->side[lane - 1];
        b.sched = column_schedule(kind, gs[i].n);
        b.xshift = gs[i].xshift;
        launch_pass(kind, gs[i].n, gs[i].emax, gs[i].lt, b);
    }
    for (int s = 0; s < S; ++s) {
        QSM_HIP(hipEventRecord(B->ev_join[slot][s], B->side[s]));
        QSM_HIP(hipStreamWaitEvent(B->stream, B->ev_join[slot][s], 0));
    }
    return QSM_OK;
}

// The relative change of iteration `it` reaches nobody: no change is below a
// tol that is not positive, and what a run reports is the last iteration's.
static bool change_unread(const qsm_tv_batch* B, size_t it) {
    return !(B->params.tol > 0.0) && it != B->params.max_iter;
}

// rec >= 0 also records the shrink pattern of iteration it-1 as checkpoint
// `rec` (unrolled adjoint).
static int enqueue_iteration(qsm_tv_batch* B, size_t it, hipEvent_t closed, int rec = -1) {
    PassArgs a = B->args(B->d_status);
    a.parity = (int)((it - 1) & 1);
    if (it == 1 && (B->method == 1 || B->plain_shrink)) {
        // The first step is x^ = f^, from g = u = 0: no z/u update comes before
        // it (src/inversion/admm.rs:76-145).  TV with t >= 0 runs the whole pass:
        // on x_0 = u = 0 its update gives 0.  (shrink(0, t < 0) is -t, and RTS
        // has x_0 != 0.)
        run_groups(P_Z_TV_SOLVE0, B->gz, a);
        run_groups(P_Y_INV, B->gy, a);
        run_groups(P_C2R_TV, B->gxc, a);
        QSM_CHECK_LAUNCH();
        return QSM_OK;
    }
    if (it >= 2) {
        a.status_rw = B->d_status;
        a.mirror = B->h_status_dev;
    }
    const bool record = rec >= 0 || B->plain_shrink;
    a.ridx = std::max(rec, 0);
    int rc;
    if ((rc = run_pass(B, 0, record ? P_R2C_TVDIV_REC : P_R2C_TVDIV, B->gx, a))) return rc;
    if (closed) QSM_HIP(hipEventRecord(closed, B->stream));
    a.status_rw = nullptr;
    a.mirror = nullptr;
    if ((rc = run_pass(B, 1, P_Y_FWD, B->gy, a))) return rc;
    if ((rc = run_pass(B, 2, B->method == 1 ? P_Z_RTS_SOLVE : P_Z_TV_SOLVE, B->gz, a))) return rc;
    if ((rc = run_pass(B, 3, P_Y_INV, B->gy, a))) return rc;
    a.no_change = change_unread(B, it) ? 1 : 0;
    if ((rc = run_pass(B, 4, P_C2R_TV, B->gxc, a))) return rc;
    QSM_CHECK_LAUNCH();
    return QSM_OK;
}

// x_0 = 0, u_{-1} = 0 (AdmmBuffers::new, src/inversion/admm.rs:39-52), then
// f^ and inv_a (prepare_admm_spectral, src/inversion/admm.rs:150-178).
static int enqueue_setup(qsm_tv_batch* B) {
    hipStream_t st = B->stream;
    if (B->method == 1) {
        // RTS (src/inversion/rts.rs:93-183): x0 = mask * Re IFFT(FFT(f) w(D)),
        // then f^ = FFT(x0) (M/rho) inv_a and inv_a.  u[0] is what the second
        // step reads as the previous dual variable.
        for (auto& V : B->h) launch_fill_zero(st, V.u[0], 3 * (size_t)V.nx * V.ny * V.nz);
        launch_status_reset(st, B->d_status, B->nvol);
        PassArgs a = B->args(nullptr);
        run_groups(B->field32 ? P_R2C_F32 : P_R2C_F64, B->gx, a);
        run_groups(P_Y_FWD, B->gy, a);
        run_groups(P_Z_FILTER, B->gz, a);
        run_groups(P_Y_INV, B->gy, a);
        run_groups(P_C2R_X0, B->gxc, a);
        run_groups(P_R2C_X0, B->gx, a);
        run_groups(P_Y_FWD, B->gy, a);
        run_groups(P_Z_RTS_SETUP, B->gz, a);
        QSM_CHECK_LAUNCH();
        return QSM_OK;
    }
    for (auto& V : B->h) {
        const size_t N = (size_t)V.nx * V.ny * V.nz;
        launch_fill_zero(st, V.x[0], N);
        launch_fill_zero(st, V.u[1], 3 * N);
        if (B->plain_shrink) launch_fill_zero(st, V.u[0], 3 * N);  // (what the second iteration reads)
    }
    launch_status_reset(st, B->d_status, B->nvol);
    PassArgs a = B->args(nullptr);
    run_groups(B->field32 ? P_R2C_F32 : P_R2C_F64, B->gx, a);
    run_groups(P_Y_FWD, B->gy, a);
    run_groups(P_Z_TV_SETUP, B->gz, a);
    QSM_CHECK_LAUNCH();
    return QSM_OK;
}

// Capture the two iteration graphs on the batch's stream.  A stream that
// cannot be captured (the legacy null stream, or one already capturing)
// leaves the batch on eager launches; nothing runs during capture.  The
// graphs hold no event: the host's "iteration closed" event is recorded
// after the replay instead (see launch_iteration).
static int build_iteration_graphs(qsm_tv_batch* B) {
    for (int s = 0; s < 2; ++s) {
        const size_t it = (size_t)s + 3;  // (it - 1) & 1 == s, it >= 2
        if (hipStreamBeginCapture(B->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            (void)hipGetLastError();
            B->graph_state = -1;
            return QSM_OK;
        }
        const int rc = enqueue_iteration(B, it, nullptr);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(B->stream, &g);
        hipError_t ei = hipSuccess;
        if (!rc && e == hipSuccess && g)
            ei = with_trim([&] { return hipGraphInstantiate(&B->gexec[s], g, nullptr, nullptr, 0); });
        if (g) (void)hipGraphDestroy(g);
        if (rc) return rc;
        if (e != hipSuccess || !g || ei != hipSuccess) {
            (void)hipGetLastError();
            for (auto& x : B->gexec)
                if (x) { (void)hipGraphExecDestroy(x); x = nullptr; }
            B->graph_state = -1;
            return QSM_OK;
        }
    }
    B->graph_state = 1;
    return QSM_OK;
}

// Iteration `it` of a run: a graph replay where available, else the eager
// launches of enqueue_iteration (the first iteration always: its kernels
// differ, and RTS starts differently; the last one where only it forms its
// relative change).  `closed` marks the point after which
// iteration it-1's convergence state is in the host mirror: eagerly right
// after the first pass of iteration it, after a replay at its end.
static int launch_iteration(qsm_tv_batch* B, size_t it, hipEvent_t closed) {
    const bool last = it == B->params.max_iter && !(B->params.tol > 0.0);
    if (it >= 2 && B->graph_state == 1 && !last) {
        QSM_HIP(hipGraphLaunch(B->gexec[(it - 1) & 1], B->stream));
        if (closed) QSM_HIP(hipEventRecord(closed, B->stream));
        return QSM_OK;
    }
    return enqueue_iteration(B, it, closed);
}

static int tv_batch_run_impl(qsm_tv_batch* B, qsm_progress_fn progress, void* user) {
    if (!B) return fail(QSM_EPARAM, "batch is null");
    hipStream_t st = B->stream;
    if (B->graph_state == 0 && B->params.max_iter >= 2) {
        int rc = build_iteration_graphs(B);
        if (rc) return rc;
    }
    std::memset(B->h_status, 0, B->nvol * sizeof(VolStatus));
    {
        int rc = enqueue_setup(B);
        if (rc) return rc;
    }

    const size_t max_iter = B->params.max_iter;
    // relative_change >= 0 (or NaN), so with tol <= 0 no iteration can stop
    // early and the host never needs to look at the device state.
    const bool can_converge = B->params.tol > 0.0;
    constexpr size_t W = qsm_tv_batch::kWindow;
    if (!progress && !can_converge) {
        for (size_t it = 1; it <= max_iter; ++it) {
            int rc = launch_iteration(B, it, nullptr);
            if (rc) return rc;
        }
        prefault(B->host_out, B->host_bytes);
        if (max_iter > 0) launch_tv_reduce(st, B->d_vols, B->nvol, B->d_status, B->h_status_dev);
    } else {
        // Iteration j is closed by the first pass of iteration j+1 (or by
        // k_tv_reduce after the last one); ev[j % W] marks that point.  Keep
        // up to W iterations in flight; report progress for iteration it+1
        // only once iteration it is known not to have converged, so the
        // callback sequence equals the reference's.
        size_t next = 1;
        if (max_iter > 0 && progress) progress(1, max_iter, user);
        for (size_t it = 1; it <= max_iter; ++it) {
            while (next <= max_iter && next <= it + W) {
                int rc = launch_iteration(B, next, next >= 2 ? B->ev[(next - 1) % W] : nullptr);
                if (rc) return rc;
                ++next;
            }
            if (it == 1) prefault(B->host_out, B->host_bytes);
            if (it == max_iter) {
                launch_tv_reduce(st, B->d_vols, B->nvol, B->d_status, B->h_status_dev);
                QSM_HIP(hipEventRecord(B->ev[it % W], st));
            }
            QSM_HIP(hipEventSynchronize(B->ev[it % W]));
            bool all_done = true;
            for (int v = 0; v < B->nvol; ++v) {
                const volatile VolStatus* hs = B->h_status + v;
                const int done = hs->done, iters = hs->iters;
                if (!(done && (size_t)iters <= it)) all_done = false;
            }
            if (all_done) {
                if (progress) progress(it, it, user);
                break;
            }
            if (it < max_iter && progress) progress(it + 1, max_iter, user);
        }
    }
    launch_tv_output(st, B->d_vols, B->lt_out, B->d_status);
    QSM_CHECK_LAUNCH();
    QSM_HIP(hipStreamSynchronize(st));
    return QSM_OK;
}

// The one volume of a host entry point: workspaces, and the field (in f32, the
// precision of the first pass) and mask uploaded.
static int host_volume_upload(HostVolume& hv, const double* field, const uint8_t* mask, size_t N) {
    int rc;
    if ((rc = dev_alloc(&hv.field, N)) || (rc = dev_alloc(&hv.chi, N)) || (rc = dev_alloc(&hv.mask, N))) return rc;
    hipError_t e = copy_to_device_f32(hv.field, field, N);
    if (e == hipSuccess) e = copy_to_device(hv.mask, mask, N);
    if (e != hipSuccess) return fail(QSM_EHIP, "hipMemcpy H2D: %s", hipGetErrorString(e));
    return QSM_OK;
}
static int host_volume_download(const HostVolume& hv, double* chi_out, size_t N) {
    const hipError_t e = copy_to_host_f32(chi_out, hv.chi, N);
    if (e != hipSuccess) return fail(QSM_EHIP, "hipMemcpy D2H: %s", hipGetErrorString(e));
    return QSM_OK;
}
static void host_volume_free(HostVolume& hv) {
    workspace_free(hv.field);
    workspace_free(hv.chi);
    workspace_free(hv.mask);
}
static qsm_tv_volume host_volume(const qsm_grid* grid, const double bdir[3]) {
    qsm_tv_volume vol{};
    vol.grid = *grid;
    for (int a = 0; a < 3; ++a) vol.bdir[a] = bdir[a];
    return vol;
}

// Event-timed copy of the iteration loop: every kernel of `iters` iterations
// is bracketed by HIP events on the batch's stream; ms_out[k] receives the
// mean duration of kernel slot k (0 r2c+div, 1 y fwd, 2 z solve, 3 y inv,
// 4 c2r).  The r2c slot includes the reduction of the previous iteration's
// relative change.  Runs the spectral setup first so the data are realistic.
static int tv_batch_profile_impl(qsm_tv_batch* B, size_t iters, double* ms_out, size_t n_out) {
    if (!B || !ms_out || n_out < 5 || iters == 0) return fail(QSM_EPARAM, "bad profile arguments");
    hipStream_t st = B->stream;
    {
        int rc = enqueue_setup(B);
        if (rc) return rc;
    }
    hipEvent_t ev[6];
    for (auto& e : ev) QSM_HIP(hipEventCreate(&e));
    double acc[5] = {0, 0, 0, 0, 0};
    PassArgs a = B->args(nullptr);
    for (size_t it = 1; it <= iters; ++it) {
        a.parity = (int)((it - 1) & 1);
        a.status_rw = it >= 2 ? B->d_status : nullptr;
        QSM_HIP(hipEventRecord(ev[0], st));
        run_groups(B->plain_shrink ? P_R2C_TVDIV_REC : P_R2C_TVDIV, B->gx, a);
        a.status_rw = nullptr;
        QSM_HIP(hipEventRecord(ev[1], st));
        run_groups(P_Y_FWD, B->gy, a);
        QSM_HIP(hipEventRecord(ev[2], st));
        run_groups(B->method == 1 ? P_Z_RTS_SOLVE : P_Z_TV_SOLVE, B->gz, a);
        QSM_HIP(hipEventRecord(ev[3], st));
        run_groups(P_Y_INV, B->gy, a);
        QSM_HIP(hipEventRecord(ev[4], st));
        a.no_change = change_unread(B, it) ? 1 : 0;
        run_groups(P_C2R_TV, B->gxc, a);
        QSM_HIP(hipEventRecord(ev[5], st));
        QSM_CHECK_LAUNCH();
        QSM_HIP(hipEventSynchronize(ev[5]));
        for (int k = 0; k < 5; ++k) {
            float ms = 0.f;
            QSM_HIP(hipEventElapsedTime(&ms, ev[k], ev[k + 1]));
            acc[k] += ms;
        }
    }
    for (auto& e : ev) (void)hipEventDestroy(e);
    for (int k = 0; k < 5; ++k) ms_out[k] = acc[k] / (double)iters;
    return QSM_OK;
}

// ============================================ unrolled TV-ADMM adjoint ====
// K iterations of tv_admm with tol = 0 (src/inversion/tv.rs:63-97) and the
// vector-Jacobian product of chi = mask * x_K with respect to the local
// field and lambda.  The forward records, for iterations 1..K-1, the shrink
// pattern q = sign(v) [|v| > lambda/rho] (one byte per component): with it
// the backward recursion is linear and needs no recomputation of the
// forward iterates.
struct qsm_tv_unrolled {
    qsm_tv_batch* B = nullptr;
    size_t K = 0;
    std::vector<int> nblk;  // x-pass blocks per volume
    std::vector<void*> allocs;
    double* d_lbar = nullptr;
    bool forward_done = false;
};

static void unrolled_free(qsm_tv_unrolled* U) {
    if (!U) return;
    if (U->B) {
        if (U->B->stream) (void)hipStreamSynchronize(U->B->stream);
        batch_free(U->B);
    }
    for (void* p : U->allocs) workspace_free(p);
    delete U;
}

static int unrolled_create_impl(const qsm_tv_volume* vols, size_t n_vols, const qsm_tv_params* params,
                                void* stream, qsm_tv_unrolled** out) {
    if (!params || !out) return fail(QSM_EPARAM, "null argument");
    qsm_tv_params p = *params;
    p.tol = 0.0;  // unrolled: exactly max_iter iterations
    qsm_tv_unrolled* U = new qsm_tv_unrolled();
    U->K = p.max_iter;
    auto cleanup = [&](int rc) { unrolled_free(U); return rc; };
    int rc = tv_batch_create_impl(vols, n_vols, &p, stream, &U->B, nullptr, nullptr, true);
    if (rc) return cleanup(rc);
    qsm_tv_batch* B = U->B;
    const size_t nrec = U->K > 1 ? U->K - 1 : 0;
    if ((rc = dev_alloc(&U->d_lbar, n_vols))) return cleanup(rc);
    U->allocs.push_back(U->d_lbar);
    for (int v = 0; v < B->nvol; ++v) {
        VolDesc& V = B->h[v];
        const size_t N = (size_t)V.nx * V.ny * V.nz;
        const int npairs = (V.ny * V.nz + 1) / 2;
        const int nb = (npairs + V.rows_x - 1) / V.rows_x;
        U->nblk.push_back(nb);
        V.adj_nblk = nb;
        if ((rc = dev_alloc(&V.ckpt, std::max<size_t>(1, nrec) * 3 * N))) return cleanup(rc);
        U->allocs.push_back(V.ckpt);
        if ((rc = dev_alloc(&V.adj_c, N))) return cleanup(rc);
        U->allocs.push_back(V.adj_c);
        for (int q = 0; q < 2; ++q) {
            if ((rc = dev_alloc(&V.adj_s[q], 3 * N))) return cleanup(rc);
            U->allocs.push_back(V.adj_s[q]);
        }
        if ((rc = dev_alloc(&V.adj_acc, N))) return cleanup(rc);
        U->allocs.push_back(V.adj_acc);
        if ((rc = dev_alloc(&V.adj_tpart, std::max<size_t>(1, nrec) * (size_t)nb))) return cleanup(rc);
        U->allocs.push_back(V.adj_tpart);
        V.adj_lbar = U->d_lbar + v;
    }
    hipError_t e = hipMemcpy(B->d_vols, B->h.data(), B->h.size() * sizeof(VolDesc), hipMemcpyHostToDevice);
    if (e != hipSuccess) return cleanup(fail(QSM_EHIP, "hipMemcpy descriptors: %s", hipGetErrorString(e)));
    *out = U;
    return QSM_OK;
}

static int unrolled_forward_impl(qsm_tv_unrolled* U) {
    if (!U) return fail(QSM_EPARAM, "handle is null");
    qsm_tv_batch* B = U->B;
    hipStream_t st = B->stream;
    std::memset(B->h_status, 0, B->nvol * sizeof(VolStatus));
    int rc = enqueue_setup(B);
    if (rc) return rc;
    for (size_t it = 1; it <= U->K; ++it) {
        if ((rc = enqueue_iteration(B, it, nullptr, it >= 2 ? (int)(it - 2) : -1))) return rc;
    }
    if (U->K > 0) launch_tv_reduce(st, B->d_vols, B->nvol, B->d_status, B->h_status_dev);
    launch_tv_output(st, B->d_vols, B->lt_out, B->d_status);
    QSM_CHECK_LAUNCH();
    QSM_HIP(hipStreamSynchronize(st));
    U->forward_done = true;
    return QSM_OK;
}

static int unrolled_backward_impl(qsm_tv_unrolled* U, const double* const* d_chi_bar,
                                  double* const* d_field_bar, double* lambda_bar) {
    if (!U || !d_chi_bar || !d_field_bar) return fail(QSM_EPARAM, "null argument");
    if (!U->forward_done) return fail(QSM_EPARAM, "backward needs a forward pass first");
    qsm_tv_batch* B = U->B;
    hipStream_t st = B->stream;
    for (int v = 0; v < B->nvol; ++v) {
        if (!d_chi_bar[v] || !d_field_bar[v]) return fail(QSM_EPARAM, "volume %d has a null pointer", v);
        B->h[v].adj_chibar = d_chi_bar[v];
        B->h[v].adj_out = d_field_bar[v];
    }
    QSM_HIP(hipMemcpyAsync(B->d_vols, B->h.data(), B->h.size() * sizeof(VolDesc), hipMemcpyHostToDevice, st));
    PassArgs a = B->args(nullptr);
    const size_t K = U->K;
    if (K == 0) {
        // chi = mask * x_0 = 0 does not depend on the field or lambda
        for (int v = 0; v < B->nvol; ++v) {
            const VolDesc& V = B->h[v];
            const size_t N = (size_t)V.nx * V.ny * V.nz;
            launch_fill_zero(st, reinterpret_cast<float*>(V.adj_out), 2 * N);
        }
        QSM_HIP(hipStreamSynchronize(st));
        if (lambda_bar)
            for (int v = 0; v < B->nvol; ++v) lambda_bar[v] = 0.0;
        return QSM_OK;
    }
    for (size_t j = K; j >= 1; --j) {
        a.parity = (int)(j & 1);
        a.ridx = (j == K) ? -1 : (int)(j - 1);
        run_groups(j == K ? P_R2C_TVADJ_FIRST : P_R2C_TVADJ, B->gx, a);
        if (j > 1) {  // c-bar_j feeds iteration j-1; c-bar_1 is not needed
            run_groups(P_Y_FWD, B->gy, a);
            run_groups(P_Z_TV_ADJ, B->gz, a);
            run_groups(P_Y_INV, B->gy, a);
            run_groups(P_C2R_ADJ, B->gxc, a);
        }
        QSM_CHECK_LAUNCH();
    }
    // field-bar = A (sum_j x-bar_j)
    run_groups(P_R2C_ACC, B->gx, a);
    run_groups(P_Y_FWD, B->gy, a);
    run_groups(P_Z_TV_APPLYA, B->gz, a);
    run_groups(P_Y_INV, B->gy, a);
    run_groups(P_C2R_F64OUT, B->gxc, a);
    launch_tv_lbar(st, B->d_vols, B->nvol, (int)(K - 1));
    QSM_CHECK_LAUNCH();
    if (lambda_bar)
        QSM_HIP(hipMemcpyAsync(lambda_bar, U->d_lbar, B->nvol * sizeof(double), hipMemcpyDeviceToHost, st));
    QSM_HIP(hipStreamSynchronize(st));
    return QSM_OK;
}

// =================================================== dipole operator ======
// field = Re IFFT(D FFT(chi)) (tests/chisep_integration.rs:18-62, kernel of
// src/kernels/dipole.rs:24-72), device pointers, f64 in and out, FP32
// transforms.  D is real and even after taking its Hermitian part, so the
// operator is self-adjoint and the adjoint entry point runs the same passes.
// zkind P_Z_DIPOLE (d_in, d_out: f64 on the device, no mask) or P_Z_FILTER
// (filter `filt` with parameter `fa`; hv: f32 field, mask and masked f32 output,
// or the phase in d_in where src_kind is P_R2C_WRAPLAP, its masked wrapped
// Laplacian); bdir may be null for filters that do not use D.
// The five passes of one spectral round trip of a single volume: R2C of
// src_kind, y, z pass zkind, inverse y, C2R pass out_kind.
// Launch tables live on the stack.
static void enqueue_round_trip(int src_kind, int zkind, int out_kind, const VolDesc& V, const PassBlocks& pb,
                               const VolDesc* d_vols, const float2* d_tw, hipStream_t st) {
    auto table = [](int blocks) {
        LaunchTable lt{};
        lt.nvol = 1;
        lt.start[0] = 0;
        lt.start[1] = blocks;
        lt.vol[0] = 0;
        return lt;
    };
    const LaunchTable tx = table(pb.xpass), txc = table(pb.cpass), ty = table(pb.ypass),
                      tz = table(pb.zpass);
    PassArgs a{};
    a.stream = st;
    a.vols = d_vols;
    a.tw = d_tw;
    a.sel = SPEC_WORK;
    a.sel2 = -1;
    a.xshift = 0;
    auto run = [&](int kind, int n, bool column, const LaunchTable& lt) {
        a.sched = column_schedule(kind, n);
        launch_pass(kind, n, emax_for(n, column), lt, a);
    };
    run(src_kind, V.nx, false, tx);
    run(P_Y_FWD, V.ny, true, ty);
    run(zkind, V.nz, true, tz);
    run(P_Y_INV, V.ny, true, ty);
    run(out_kind, V.nx, false, txc);
}

static int spectral_apply(int zkind, int filt, double fa, const double* d_in, const qsm_grid* grid,
                          const double bdir_in[3], double* d_out, void* stream, int src_kind = P_R2C_F64,
                          const HostVolume* hv = nullptr) {
    static const double z_axis[3] = {0.0, 0.0, 1.0};
    const double* bdir = bdir_in ? bdir_in : z_axis;
    if (!hv && (!d_in || !grid || !d_out)) return fail(QSM_EPARAM, "null argument");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const double bn = std::sqrt(bdir[0] * bdir[0] + bdir[1] * bdir[1] + bdir[2] * bdir[2]);
    if (!(bn > 0)) return fail(QSM_EPARAM, "B0 direction has zero length");
    VolDesc V;
    std::memset(&V, 0, sizeof V);
    TwiddleBank tb;
    PassBlocks pb = fill_geometry(V, *grid, tb, pair_rows(*grid), ROWS_SINGLE);
    V.bx = bdir[0] / bn; V.by = bdir[1] / bn; V.bz = bdir[2] / bn;
    V.field = d_in;
    V.adj_out = d_out;
    if (hv) {
        V.vs_local = hv->field;
        V.mask = hv->mask;
        V.x[0] = hv->chi;
    }
    V.filt = filt;
    V.filt_a = fa;
    const size_t Nh = (size_t)V.nxh * V.ny * V.nz;
    std::vector<void*> allocs;
    float2* d_tw = nullptr;
    VolDesc* d_vols = nullptr;
    hipStream_t st = (hipStream_t)stream;
    bool own = false;
    auto done = [&](int code) {
        if (st) (void)hipStreamSynchronize(st);
        for (void* p : allocs) workspace_free(p);
        if (own) stream_give(st);
        return code;
    };
    if ((rc = dev_alloc(&V.spec[SPEC_WORK], Nh))) return done(rc);
    allocs.push_back(V.spec[SPEC_WORK]);
    {
        void* block = nullptr;
        rc = upload_plan(&V, 1, tb, &block, &d_vols, &d_tw);
        if (block) allocs.push_back(block);
        if (rc) return done(rc);
    }
    if (!st) {
        hipError_t e = stream_take(&st);
        if (e != hipSuccess) { st = nullptr; return done(fail(QSM_EHIP, "hipStreamCreate: %s", hipGetErrorString(e))); }
        own = true;
    }
    enqueue_round_trip(src_kind, zkind, hv ? P_C2R_X0 : P_C2R_F64OUT, V, pb, d_vols, d_tw, st);
    hipError_t le = hipGetLastError();
    if (le != hipSuccess) return done(fail(QSM_EHIP, "kernel launch: %s", hipGetErrorString(le)));
    if (hv) prefault(hv->out, hv->n * sizeof(double));
    hipError_t se = hipStreamSynchronize(st);
    if (se != hipSuccess) return done(fail(QSM_EHIP, "hipStreamSynchronize: %s", hipGetErrorString(se)));
    return done(QSM_OK);
}

// ========================================================= V-SHARP batch ==
// Voxels of the wrapped sphere of src/kernels/smv.rs:19-67, counted over the
// sphere's bounding box only (same coordinates and the same f64 operation
// order as the kernel, so the count equals the reference's `count`).
static double sphere_count(const qsm_grid& g, double radius) {
#pragma clang fp contract(off)
    const double r2 = radius * radius;
    auto coords = [&](size_t n, double vs, std::vector<double>& out) {
        const double lim = std::fabs(radius) / vs + 1.0;
        for (size_t i = 0; i < n; ++i) {
            double c = (i <= n / 2) ? (double)i : (double)((long long)i - (long long)n);
            if (std::fabs(c) <= lim) out.push_back(c * vs);
        }
    };
    std::vector<double> xs, ys, zs;
    coords(g.nx, g.vsx, xs);
    coords(g.ny, g.vsy, ys);
    coords(g.nz, g.vsz, zs);
    double count = 0.0;
    for (double dz : zs)
        for (double dy : ys)
            for (double dx : xs) {
                volatile double d2 = dx * dx;
                d2 = d2 + dy * dy;
                d2 = d2 + dz * dz;
                if (d2 <= r2) count += 1.0;
            }
    return count;
}

struct qsm_vsharp_batch {
    int nvol = 0;
    std::vector<VolDesc> h;
    VolDesc* d_vols = nullptr;
    float2* d_tw = nullptr;
    double* d_radii = nullptr;
    std::vector<double> radii;  // processing order (descending)
    double threshold = 0.05;
    bool sharp = false;         // one radius: sharp_core semantics
    bool field32 = false;       // the field is in VolDesc::vs_local, in f32, until that is cleared (host entry point)
    void* host_out = nullptr;   // its result array, made ready while the device works
    size_t host_bytes = 0;
    Groups gx, grows, gy, gy2, gz;   // passes grouped by axis length
    LaunchTable lt_init{};
    std::vector<void*> allocs;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    PassArgs args() const {
        PassArgs a{};
        a.stream = stream;
        a.vols = d_vols;
        a.tw = d_tw;
        a.status = nullptr;
        a.sel = SPEC_WORK;
        a.sel2 = -1;
        return a;
    }
};

static void vs_free(qsm_vsharp_batch* b) {
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    for (void* p : b->allocs) workspace_free(p);
    if (b->own_stream && b->stream) stream_give(b->stream);
    delete b;
}

static int vs_create_impl(const qsm_vsharp_volume* vols, size_t n_vols, const double* radii,
                          size_t n_radii, double threshold, void* stream, qsm_vsharp_batch** out,
                          const HostVolume* io = nullptr) {
    if (!vols || !out || (n_radii && !radii)) return fail(QSM_EPARAM, "null argument");
    if (n_vols == 0 || n_vols > (size_t)kMaxVolumes)
        return fail(QSM_EPARAM, "batch size %zu outside 1..%d", n_vols, kMaxVolumes);
    if (n_radii == 0) return fail(QSM_EPARAM, "at least one radius is required for a batch");
    for (size_t r = 0; r < n_radii; ++r)
        if (std::isnan(radii[r])) return fail(QSM_EPARAM, "radius %zu is NaN", r);
    for (size_t v = 0; v < n_vols; ++v) {
        int rc = validate_grid(&vols[v].grid);
        if (rc) return rc;
        if (!io && (!vols[v].d_field || !vols[v].d_mask || !vols[v].d_local || !vols[v].d_mask_out))
            return fail(QSM_EPARAM, "volume %zu has a null device pointer", v);
    }
    qsm_vsharp_batch* B = new qsm_vsharp_batch();
    auto cleanup = [&](int rc) { vs_free(B); return rc; };
    B->nvol = (int)n_vols;
    B->threshold = threshold;
    // src/bgremove/vsharp.rs:114-116: sort descending (stable)
    B->radii.assign(radii, radii + n_radii);
    std::stable_sort(B->radii.begin(), B->radii.end(), [](double a, double b) { return b < a; });
    B->sharp = (n_radii == 1);
    const int R = (int)n_radii;
    B->h.resize(n_vols);
    TwiddleBank tb;
    std::vector<int> lx, ly, lz, bx, brows, by, by2, bz, bi;
    std::map<size_t, size_t> pairs = length_pairs(vols, n_vols);
    int rc;
    if ((rc = dev_alloc(&B->d_radii, (size_t)R * (1 + n_vols)))) return cleanup(rc);
    B->allocs.push_back(B->d_radii);
    std::vector<double> host_tab((size_t)R * (1 + n_vols));
    for (int r = 0; r < R; ++r) host_tab[r] = B->radii[r];
    for (size_t v = 0; v < n_vols; ++v) {
        VolDesc& V = B->h[v];
        std::memset(&V, 0, sizeof V);
        // (the selection pass has twice as many rows as the others pair-rows)
        PassBlocks pb = fill_geometry(V, vols[v].grid, tb, 2 * pairs[vols[v].grid.nx], ROWS_SINGLE);
        V.field = vols[v].d_field;
        V.mask = vols[v].d_mask;
        V.out = vols[v].d_local;
        V.mask_out = vols[v].d_mask_out;
        if (io) {
            V.mask = io->mask;
            V.out32 = io->chi;
            B->field32 = true;
        }
        V.vs_threshold = threshold;
        V.vs_radii = B->d_radii;
        V.vs_counts = B->d_radii + (size_t)R * (1 + v);
        for (int r = 0; r < R; ++r) host_tab[(size_t)R * (1 + v) + r] = sphere_count(vols[v].grid, B->radii[r]);
        const int nrows = V.ny * V.nz;
        lx.push_back(V.nx); bx.push_back(pb.xpass);
        brows.push_back((nrows + V.rows_x - 1) / V.rows_x);
        ly.push_back(V.ny); by.push_back(pb.ypass); by2.push_back(2 * pb.ypass);
        lz.push_back(V.nz); bz.push_back(pb.zpass);
        bi.push_back(pb.out);
        const size_t N = (size_t)V.nx * V.ny * V.nz;
        const size_t Nh = (size_t)V.nxh * V.ny * V.nz;
        for (int sidx = 0; sidx < SPEC_COUNT; ++sidx) {
            if ((rc = dev_alloc(&V.spec[sidx], Nh))) return cleanup(rc);
            B->allocs.push_back(V.spec[sidx]);
        }
        // S^ of the largest sphere; 2 nz more for the Nyquist plane's doubly packed columns
        if ((rc = dev_alloc(&V.vs_sfirst, Nh + 2 * (size_t)V.nz))) return cleanup(rc);
        B->allocs.push_back(V.vs_sfirst);
        if ((rc = dev_alloc(&V.vs_local, N))) return cleanup(rc);
        B->allocs.push_back(V.vs_local);
        if ((rc = dev_alloc(&V.vs_final, N))) return cleanup(rc);
        B->allocs.push_back(V.vs_final);
    }
    B->gx = make_groups(lx, bx, false);
    B->grows = make_groups(lx, brows, false);
    B->gy = make_groups(ly, by, true);
    B->gy2 = make_groups(ly, by2, true);
    B->gz = make_groups(lz, bz, true);
    B->lt_init = identity_table(bi);
    {
        void* block = nullptr;
        rc = upload_plan(B->h.data(), n_vols, tb, &block, &B->d_vols, &B->d_tw);
        if (block) B->allocs.push_back(block);
        if (rc) return cleanup(rc);
    }
    if (stream) {
        B->stream = (hipStream_t)stream;
    } else {
        hipError_t e = stream_take(&B->stream);
        if (e != hipSuccess) { B->stream = nullptr; return cleanup(fail(QSM_EHIP, "hipStreamCreate: %s", hipGetErrorString(e))); }
        B->own_stream = true;
    }
    hipError_t e3 = hipMemcpy(B->d_radii, host_tab.data(), host_tab.size() * sizeof(double), hipMemcpyHostToDevice);
    if (e3 != hipSuccess) return cleanup(fail(QSM_EHIP, "hipMemcpy of plan tables failed"));
    *out = B;
    return QSM_OK;
}

static int vs_run_impl(qsm_vsharp_batch* B, qsm_progress_fn progress, void* user) {
    if (!B) return fail(QSM_EPARAM, "batch is null");
    hipStream_t st = B->stream;
    const int R = (int)B->radii.size();
    const double delta = 1.0 - std::sqrt(1e-7);  // src/bgremove/vsharp.rs:129
    // F^ = FFT(field) (vsharp.rs:117-122), M^ = FFT(mask) once for all radii
    PassArgs a = B->args();
    a.sel = SPEC_A;
    run_groups(B->field32 ? P_R2C_F32 : P_R2C_F64, B->gx, a);
    run_groups(P_Y_FWD, B->gy, a);
    run_groups(P_Z_VS_FWD, B->gz, a);
    a.sel = SPEC_B;
    run_groups(P_R2C_U8, B->gx, a);
    run_groups(P_Y_FWD, B->gy, a);
    run_groups(P_Z_VS_FWD, B->gz, a);
    launch_vs_init(st, B->d_vols, B->lt_init);
    QSM_CHECK_LAUNCH();
    a.sel = SPEC_WORK;
    a.delta = delta;
    for (int r = 0; r < R; ++r) {
        if (progress) {
            // report radius r+1 once radius r has finished on the device
            if (r > 0) QSM_HIP(hipStreamSynchronize(st));
            if (B->sharp) progress(1, 1, user);           // vsharp.rs:103-108
            else progress((size_t)r + 1, (size_t)R, user); // vsharp.rs:134
        }
        a.ridx = r;
        a.first = (r == 0) ? 1 : 0;
        a.sel2 = -1;
        run_groups(P_R2C_SPHERE, B->gx, a);
        run_groups(P_Y_FWD, B->gy, a);
        run_groups(P_Z_VS_RADIUS, B->gz, a);
        a.sel2 = SPEC_C;
        run_groups(P_Y_INV, B->gy2, a);
        a.sel2 = -1;
        run_groups(P_C2R_VS_SELECT, B->grows, a);
        QSM_CHECK_LAUNCH();
    }
    // deconvolution with the largest kernel (vsharp.rs:180-196 / sharp.rs:105-131)
    a.divide = B->sharp ? 1 : 0;
    run_groups(P_R2C_F32, B->gx, a);
    run_groups(P_Y_FWD, B->gy, a);
    run_groups(P_Z_VS_DECONV, B->gz, a);
    run_groups(P_Y_INV, B->gy, a);
    run_groups(P_C2R_VS_OUT, B->gx, a);
    QSM_CHECK_LAUNCH();
    prefault(B->host_out, B->host_bytes);
    QSM_HIP(hipStreamSynchronize(st));
    return QSM_OK;
}

// Host-pointer V-SHARP with explicit radii (src/bgremove/vsharp.rs:88-199).
static int vsharp_host(const double* field, const uint8_t* mask, const qsm_grid* grid,
                       const double* radii, size_t n_radii, double threshold,
                       qsm_progress_fn progress, void* user, double* local_out, uint8_t* mask_out) {
    if (!field || !mask || !grid || !local_out || !mask_out || (n_radii && !radii))
        return fail(QSM_EPARAM, "null argument");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const size_t N = grid->nx * grid->ny * grid->nz;
    if (n_radii == 0) {  // vsharp.rs:98-100
        std::fill(local_out, local_out + N, 0.0);
        std::memcpy(mask_out, mask, N);
        return QSM_OK;
    }
    HostVolume hv;
    uint8_t* d_mo = nullptr;
    qsm_vsharp_batch* B = nullptr;
    auto done = [&](int code) {
        if (B) vs_free(B);
        host_volume_free(hv);
        workspace_free(d_mo);
        return code;
    };
    if ((rc = dev_alloc(&hv.chi, N)) || (rc = dev_alloc(&hv.mask, N)) || (rc = dev_alloc(&d_mo, N))) return done(rc);
    qsm_vsharp_volume vol{};
    vol.grid = *grid;
    vol.d_mask_out = d_mo;
    if ((rc = vs_create_impl(&vol, 1, radii, n_radii, threshold, nullptr, &B, &hv))) return done(rc);
    B->host_out = local_out;
    B->host_bytes = N * sizeof(double);
    hipError_t e = copy_to_device_f32(B->h[0].vs_local, field, N);
    if (e == hipSuccess) e = copy_to_device(hv.mask, mask, N);
    if (e != hipSuccess) return done(fail(QSM_EHIP, "hipMemcpy H2D: %s", hipGetErrorString(e)));
    if ((rc = vs_run_impl(B, progress, user))) return done(rc);
    if ((rc = host_volume_download(hv, local_out, N))) return done(rc);
    e = copy_to_host(mask_out, d_mo, N);
    if (e != hipSuccess) return done(fail(QSM_EHIP, "hipMemcpy D2H: %s", hipGetErrorString(e)));
    return done(QSM_OK);
}

// src/bgremove/vsharp.rs:70-82.  A non-positive step would never terminate
// in the reference; it is rejected instead.
static int vsharp_radii(const qsm_vsharp_params* p, std::vector<double>& radii) {
    if (!(p->min_radius > 0.0))
        return fail(QSM_EPARAM, "min_radius must be > 0 (it is the step between radii)");
    if (std::isnan(p->max_radius)) return fail(QSM_EPARAM, "max_radius is NaN");
    double r = p->max_radius;
    const double step = p->min_radius;
    while (r >= step) {
        radii.push_back(r);
        r -= step;
        if (radii.size() > 100000) return fail(QSM_EPARAM, "too many radii");
    }
    if (radii.empty()) radii.push_back(p->max_radius);
    return QSM_OK;
}

// ====================================================== extern "C" API ====
extern "C" {

void qsm_tv_params_default(qsm_tv_params* p) {
    if (!p) return;
    p->lambda = 2e-4;  // src/inversion/tv.rs:34-43
    p->rho = 2e-2;
    p->tol = 1e-3;
    p->max_iter = 250;
}

void qsm_vsharp_params_default(qsm_vsharp_params* p) {
    if (!p) return;
    p->threshold = 0.05;  // src/bgremove/vsharp.rs:31-39
    p->max_radius = 12.0;
    p->min_radius = 1.0;
}

const char* qsm_last_error_message(void) { return g_err.c_str(); }

int qsm_fft_length_supported(size_t n) { return length_ok(n) ? 1 : 0; }

int qsm_backend_info(char* buf, size_t len) {
    if (!buf || len == 0) return fail(QSM_EPARAM, "null buffer");
    int dev = 0;
    hipDeviceProp_t prop;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) {
        snprintf(buf, len, "qsm_gpu (gfx950 build); no HIP device: %s", hipGetErrorString(e));
        return QSM_OK;
    }
    snprintf(buf, len, "qsm_gpu gfx950 build on %s (%s), %d CUs, %.1f GiB HBM", prop.name,
             prop.gcnArchName, prop.multiProcessorCount, prop.totalGlobalMem / 1073741824.0);
    return QSM_OK;
}

int qsm_tv_batch_create(const qsm_tv_volume* vols, size_t n_vols, const qsm_tv_params* params,
                        void* stream, qsm_tv_batch** out) {
    g_err.clear();
    return tv_batch_create_impl(vols, n_vols, params, stream, out);
}

int qsm_tv_batch_run(qsm_tv_batch* batch, qsm_progress_fn progress, void* user) {
    g_err.clear();
    return tv_batch_run_impl(batch, progress, user);
}

int qsm_set_fft_schedule(int mode) {
    g_err.clear();
    if (mode < 0 || mode > 3) return fail(QSM_EPARAM, "schedule mode must be 0, 1, 2 or 3");
    g_sched_mode.store(mode);
    return QSM_OK;
}

int qsm_fft_schedule(int axis, int n, int* sched) {
    g_err.clear();
    if (!sched || (axis != 1 && axis != 2)) return fail(QSM_EPARAM, "axis must be 1 (y) or 2 (z)");
    if (n <= 0 || n > kMaxAxis || !qsmfft::col2_ok(n)) {
        *sched = 1;  // only the staged transform exists for this length
        return QSM_OK;
    }
    const int mode = g_sched_mode.load();
    if (mode == 1 || mode == 2) {
        *sched = mode - 1;
        return QSM_OK;
    }
    if (mode == 0) {
        *sched = fixed_schedule(axis - 1, n);
        return QSM_OK;
    }
    std::lock_guard<std::mutex> lk(g_sched_mu);
    *sched = g_sched_tab[axis - 1][n];
    return QSM_OK;
}

int qsm_tv_batch_set_graphs(qsm_tv_batch* B, int enable) {
    g_err.clear();
    if (!B) return fail(QSM_EPARAM, "batch is null");
    if (!enable) {
        for (auto& g : B->gexec)
            if (g) { (void)hipGraphExecDestroy(g); g = nullptr; }
        B->graph_state = -1;
    } else if (B->graph_state == -1) {
        B->graph_state = 0;  // captured at the next run
    }
    return QSM_OK;
}

int qsm_tv_batch_status(const qsm_tv_batch* B, size_t v, size_t* iters, double* rel) {
    if (!B || v >= (size_t)B->nvol) return fail(QSM_EPARAM, "bad batch or volume index");
    VolStatus s;
    hipError_t e = hipMemcpy(&s, B->d_status + v, sizeof s, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fail(QSM_EHIP, "hipMemcpy status: %s", hipGetErrorString(e));
    if (iters) *iters = (size_t)s.iters;
    if (rel) *rel = s.rel;
    return QSM_OK;
}

void qsm_tv_batch_destroy(qsm_tv_batch* batch) { batch_free(batch); }

int qsm_tv_batch_profile(qsm_tv_batch* batch, size_t iters, double* ms_out, size_t n_out) {
    g_err.clear();
    return tv_batch_profile_impl(batch, iters, ms_out, n_out);
}

int qsm_tv_admm_ex(const double* local_field, const uint8_t* mask, const qsm_grid* grid,
                   const double bdir[3], const qsm_tv_params* params, qsm_progress_fn progress,
                   void* user, double* chi_out, size_t* iters_out, double* rel_out) {
    g_err.clear();
    if (!local_field || !mask || !grid || !bdir || !params || !chi_out)
        return fail(QSM_EPARAM, "null argument");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const size_t N = grid->nx * grid->ny * grid->nz;
    HostVolume hv;
    qsm_tv_batch* B = nullptr;
    auto done = [&](int code) {
        if (B) batch_free(B);
        host_volume_free(hv);
        return code;
    };
    if ((rc = host_volume_upload(hv, local_field, mask, N))) return done(rc);
    const qsm_tv_volume vol = host_volume(grid, bdir);
    if ((rc = tv_batch_create_impl(&vol, 1, params, nullptr, &B, nullptr, &hv))) return done(rc);
    B->graph_state = -1;  // run once: capturing the graphs costs more than they save
    B->host_out = chi_out;
    B->host_bytes = N * sizeof(double);
    if ((rc = tv_batch_run_impl(B, progress, user))) return done(rc);
    if ((rc = host_volume_download(hv, chi_out, N))) return done(rc);
    if (iters_out || rel_out) {
        size_t it = 0;
        double rel = 0;
        if ((rc = qsm_tv_batch_status(B, 0, &it, &rel))) return done(rc);
        if (iters_out) *iters_out = it;
        if (rel_out) *rel_out = rel;
    }
    return done(QSM_OK);
}

int qsm_tv_admm(const double* local_field, const uint8_t* mask, const qsm_grid* grid,
                const double bdir[3], const qsm_tv_params* params, qsm_progress_fn progress,
                void* user, double* chi_out) {
    return qsm_tv_admm_ex(local_field, mask, grid, bdir, params, progress, user, chi_out, nullptr,
                          nullptr);
}

int qsm_run_dipole_inversion(const double* local_field_ppm, size_t field_len, const uint8_t* mask,
                             size_t mask_len, const qsm_scan_metadata* md,
                             qsm_inversion_algorithm algorithm, const qsm_tv_params* tv_params,
                             qsm_progress_fn progress, void* user, double* chi_out) {
    g_err.clear();
    if (!md) return fail(QSM_EPARAM, "metadata is null");
    const size_t n = md->nx * md->ny * md->nz;
    // src/pipeline/inversion.rs:36-45
    if (field_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, field_len);
    if (mask_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, mask_len);
    if (algorithm == QSM_INV_TGV || algorithm == QSM_INV_QSMART)
        return fail(QSM_ECONFIG, "invalid config: %s should use run_tgv or run_qsmart",
                    algorithm == QSM_INV_TGV ? "Tgv" : "Qsmart");
    qsm_inversion_config cfg;
    qsm_inversion_config_default(&cfg);
    cfg.algorithm = algorithm;
    if (tv_params) cfg.tv = *tv_params;
    return qsm_run_dipole_inversion_cfg(local_field_ppm, field_len, mask, mask_len, md, &cfg, progress,
                                        user, chi_out);
}

int qsm_tv_unrolled_create(const qsm_tv_volume* vols, size_t n_vols, const qsm_tv_params* params,
                           void* stream, qsm_tv_unrolled** out) {
    g_err.clear();
    return unrolled_create_impl(vols, n_vols, params, stream, out);
}

int qsm_tv_unrolled_forward(qsm_tv_unrolled* h) {
    g_err.clear();
    return unrolled_forward_impl(h);
}

int qsm_tv_unrolled_backward(qsm_tv_unrolled* h, const double* const* d_chi_bar,
                             double* const* d_field_bar, double* lambda_bar) {
    g_err.clear();
    return unrolled_backward_impl(h, d_chi_bar, d_field_bar, lambda_bar);
}

void qsm_tv_unrolled_destroy(qsm_tv_unrolled* h) { unrolled_free(h); }

int qsm_dipole_forward(const double* d_chi, const qsm_grid* grid, const double bdir[3], double* d_field,
                       void* stream) {
    g_err.clear();
    return spectral_apply(P_Z_DIPOLE, 0, 0.0, d_chi, grid, bdir, d_field, stream);
}

int qsm_dipole_adjoint(const double* d_field, const qsm_grid* grid, const double bdir[3], double* d_chi,
                       void* stream) {
    g_err.clear();
    return spectral_apply(P_Z_DIPOLE, 0, 0.0, d_field, grid, bdir, d_chi, stream);
}

// ------------------------------------- dipole operator, no allocation ----
// Workspace of qsm_dipole_forward_noalloc in a file-scope device array: the
// volume descriptor, the FFT tables of three lengths and one half spectrum.  Each device holds its own copy until the process ends.  Host
// code never passes `scratch` itself to a kernel or a copy: its device
// address comes from hipGetSymbolAddress, once per device.
namespace {
constexpr size_t kScratchDescBytes = 4096;
// three axes, each at most a length-1024 table with a chirp and its filter, or
// a length-512 table with two dense tables
constexpr size_t kScratchTwBytes =
    sizeof(float2) * 3 * (2 * kMaxLen + kMaxChirpLen + 2 * (size_t)qsmfft::dense_table_len(qsmfft::kMaxDenseRadix));
constexpr size_t kScratchSpecOff = 1 << 20;
constexpr size_t kScratchSpecBytes = (size_t)72 << 20;
constexpr size_t kScratchBytes = kScratchSpecOff + kScratchSpecBytes;
static_assert(sizeof(VolDesc) <= kScratchDescBytes, "descriptor does not fit its scratch slot");
static_assert(kScratchDescBytes + kScratchTwBytes <= kScratchSpecOff, "twiddles overlap the spectrum");
constexpr int kScratchMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchMaxDevices] = {};
}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on the current device (looked up on the first
// call on each device).
static int scratch_address(unsigned char** out) {
    int dev = 0;
    QSM_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kScratchMaxDevices) return fail(QSM_EHIP, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(QSM_EHIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = static_cast<unsigned char*>(g_scratch_ptr[dev]);
    return QSM_OK;
}

static int dipole_noalloc_impl(const double* d_chi, const qsm_grid* grid, const double bdir[3],
                               double* d_field, void* stream) {
    if (!d_chi || !grid || !bdir || !d_field) return fail(QSM_EPARAM, "null argument");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const double bn = std::sqrt(bdir[0] * bdir[0] + bdir[1] * bdir[1] + bdir[2] * bdir[2]);
    if (!(bn > 0)) return fail(QSM_EPARAM, "B0 direction has zero length");
    VolDesc V;
    std::memset(&V, 0, sizeof V);
    TwiddleBank tb;
    PassBlocks pb = fill_geometry(V, *grid, tb, pair_rows(*grid), ROWS_SINGLE);
    const size_t spec_bytes = (size_t)V.nxh * V.ny * V.nz * sizeof(float2);
    if (spec_bytes > kScratchSpecBytes)
        return fail(QSM_EPARAM,
                    "volume %zux%zux%zu needs %zu bytes of spectrum workspace; the fixed scratch of "
                    "qsm_dipole_forward_noalloc holds %zu (use qsm_dipole_forward)",
                    grid->nx, grid->ny, grid->nz, spec_bytes, kScratchSpecBytes);
    unsigned char* base = nullptr;
    if ((rc = scratch_address(&base))) return rc;
    VolDesc* d_vols = reinterpret_cast<VolDesc*>(base);
    float2* d_tw = reinterpret_cast<float2*>(base + kScratchDescBytes);
    V.bx = bdir[0] / bn; V.by = bdir[1] / bn; V.bz = bdir[2] / bn;
    V.field = d_chi;
    V.adj_out = d_field;
    V.spec[SPEC_WORK] = reinterpret_cast<float2*>(base + kScratchSpecOff);
    hipStream_t st = (hipStream_t)stream;
    // The R2C pass writes the whole spectrum, so nothing needs clearing.
    QSM_HIP(hipMemcpyAsync(d_vols, &V, sizeof V, hipMemcpyHostToDevice, st));
    QSM_HIP(hipMemcpyAsync(d_tw, tb.host.data(), tb.host.size() * sizeof(float2), hipMemcpyHostToDevice, st));
    enqueue_round_trip(P_R2C_F64, P_Z_DIPOLE, P_C2R_F64OUT, V, pb, d_vols, d_tw, st);
    QSM_CHECK_LAUNCH();
    // the host-side tables above live on this stack frame: wait before returning
    QSM_HIP(hipStreamSynchronize(st));
    return QSM_OK;
}

int qsm_dipole_forward_noalloc(const double* d_chi, const qsm_grid* grid, const double bdir[3],
                               double* d_field, void* stream) {
    g_err.clear();
    try {
        return dipole_noalloc_impl(d_chi, grid, bdir, d_field, stream);
    } catch (const std::bad_alloc&) {  // (the tables, before any device work)
        return QSM_ENOMEM;
    }
}

// Host-array wrapper of a closed-form inversion (filter kind, parameter).
static int filter_host(int filt, double fa, const double* field, const uint8_t* mask,
                       const qsm_grid* grid, const double bdir[3], double* chi_out,
                       int src_kind = P_R2C_F64) {
    if (!field || !mask || !grid || (!bdir && src_kind == P_R2C_F64) || !chi_out)
        return fail(QSM_EPARAM, "null argument");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const size_t N = grid->nx * grid->ny * grid->nz;
    // the wrapped Laplacian takes the phase in f64; every other source is f32 on
    // the device, and so is the output
    double* d_f64 = nullptr;
    HostVolume hv;
    auto done = [&](int code) {
        workspace_free(d_f64);
        host_volume_free(hv);
        return code;
    };
    const bool wrapped = src_kind == P_R2C_WRAPLAP;
    hv.out = chi_out;
    hv.n = N;
    if (wrapped) {
        if ((rc = dev_alloc(&d_f64, N)) || (rc = dev_alloc(&hv.chi, N)) || (rc = dev_alloc(&hv.mask, N))) return done(rc);
        hipError_t e = copy_to_device(d_f64, field, N * sizeof(double));
        if (e == hipSuccess) e = copy_to_device(hv.mask, mask, N);
        if (e != hipSuccess) return done(fail(QSM_EHIP, "hipMemcpy H2D: %s", hipGetErrorString(e)));
    } else if ((rc = host_volume_upload(hv, field, mask, N))) {
        return done(rc);
    }
    if ((rc = spectral_apply(P_Z_FILTER, filt, fa, d_f64, grid, bdir, nullptr, nullptr,
                             wrapped ? P_R2C_WRAPLAP : P_R2C_F32, &hv)))
        return done(rc);
    if ((rc = host_volume_download(hv, chi_out, N))) return done(rc);
    return done(QSM_OK);
}

// laplacian_unwrap, src/unwrap/laplacian.rs:135-161: Poisson solve of the
// masked wrapped Laplacian, masked.
int qsm_laplacian_unwrap(const double* phase, const uint8_t* mask, const qsm_grid* grid, double* out) {
    g_err.clear();
    return filter_host(6, 0.0, phase, mask, grid, nullptr, out, P_R2C_WRAPLAP);
}

// nltv, src/inversion/nltv.rs:63-133, on one volume: TV's kernels with
// weighted thresholds, a weight pass and a boundary step between Newton
// rounds.  The host synchronises after every step when it needs to know
// about convergence (tol > 0) or report progress.
void qsm_nltv_params_default(qsm_nltv_params* p) {
    if (!p) return;  // src/inversion/nltv.rs:38-49
    p->lambda = 1e-3;
    p->mu = 1.0;
    p->tol = 1e-3;
    p->max_iter = 250;
    p->newton_iter = 10;
}

int qsm_nltv(const double* local_field, const uint8_t* mask, const qsm_grid* grid, const double bdir[3],
             const qsm_nltv_params* params, qsm_progress_fn progress, void* user, double* chi_out) {
    g_err.clear();
    if (!local_field || !mask || !grid || !bdir || !params || !chi_out)
        return fail(QSM_EPARAM, "null argument");
    if (!(params->lambda > 0)) return fail(QSM_EPARAM, "NLTV needs lambda > 0 (rho = 100 lambda)");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const size_t N = grid->nx * grid->ny * grid->nz;
    HostVolume hv;
    qsm_tv_batch* B = nullptr;
    std::vector<void*> extra;
    auto done = [&](int code) {
        if (B) batch_free(B);
        for (void* p : extra) workspace_free(p);
        host_volume_free(hv);
        return code;
    };
    if ((rc = host_volume_upload(hv, local_field, mask, N))) return done(rc);
    const qsm_tv_volume vol = host_volume(grid, bdir);
    qsm_tv_params tp;
    tp.lambda = params->lambda;
    tp.rho = 100.0 * params->lambda;  // src/inversion/nltv.rs:75
    tp.tol = params->tol;
    tp.max_iter = params->max_iter;
    if ((rc = tv_batch_create_impl(&vol, 1, &tp, nullptr, &B, nullptr, &hv))) return done(rc);
    VolDesc& V = B->h[0];
    V.filt_b = params->mu;
    const int nb = (int)((N + qsmfft::kThreads * 4 - 1) / (qsmfft::kThreads * 4));
    for (int q = 0; q < 2; ++q) {
        if ((rc = dev_alloc(&V.nltv_w[q], N))) return done(rc);
        extra.push_back(V.nltv_w[q]);
    }
    if ((rc = dev_alloc(&V.nltv_wnorm, 2))) return done(rc);
    extra.push_back(V.nltv_wnorm);
    if ((rc = dev_alloc(&V.nltv_wpart, (size_t)nb))) return done(rc);
    extra.push_back(V.nltv_wpart);
    hipStream_t st = B->stream;
    QSM_HIP(hipMemcpy(B->d_vols, B->h.data(), sizeof(VolDesc), hipMemcpyHostToDevice));
    std::memset(B->h_status, 0, sizeof(VolStatus));
    if ((rc = enqueue_setup(B))) return done(rc);
    launch_nltv_init(st, B->d_vols, B->lt_out);
    const bool sync_each = progress != nullptr || params->tol > 0.0;
    const size_t total = params->max_iter * params->newton_iter;
    size_t S = 0, current = 0;
    int cw = 0;
    hipEvent_t ev = B->ev[0];
    for (size_t newton = 0; newton < params->newton_iter; ++newton) {
        for (size_t it = 1; it <= params->max_iter; ++it) {
            ++current;
            if (progress) progress(current, total, user);
            ++S;
            PassArgs a = B->args(B->d_status);
            a.parity = (int)((S - 1) & 1);
            if (newton > 0 && it == 1) {
                launch_nltv_weights(st, B->d_vols, B->lt_out, a.parity, cw ^ 1);
                launch_nltv_wmax(st, B->d_vols, 1, nb, cw ^ 1);
                PassArgs b = a;
                b.status_rw = B->d_status;
                b.ridx = cw;
                run_groups(P_R2C_NLTV_BND, B->gx, b);
                launch_status_clear_done(st, B->d_status, 1);
                cw ^= 1;
            } else {
                a.ridx = cw;
                run_groups(P_R2C_TVDIV_W, B->gx, a);
            }
            run_groups(P_Y_FWD, B->gy, a);
            run_groups(P_Z_TV_SOLVE, B->gz, a);
            run_groups(P_Y_INV, B->gy, a);
            run_groups(P_C2R_TV, B->gxc, a);
            launch_tv_reduce(st, B->d_vols, 1, B->d_status, B->h_status_dev);
            QSM_CHECK_LAUNCH();
            if (sync_each) {
                QSM_HIP(hipEventRecord(ev, st));
                QSM_HIP(hipEventSynchronize(ev));
                const volatile VolStatus* hs = B->h_status;
                if (hs->done) break;  // src/inversion/nltv.rs:105-107
            }
        }
    }
    launch_tv_output(st, B->d_vols, B->lt_out, B->d_status);
    QSM_CHECK_LAUNCH();
    QSM_HIP(hipStreamSynchronize(st));
    if ((rc = host_volume_download(hv, chi_out, N))) return done(rc);
    return done(QSM_OK);
}

void qsm_tkd_params_default(qsm_tkd_params* p) {
    if (p) p->threshold = 0.15;  // src/inversion/tkd.rs:29-33
}

void qsm_tikhonov_params_default(qsm_tikhonov_params* p) {
    if (!p) return;
    p->lambda = 0.01;  // src/inversion/tikhonov.rs:45-49
    p->reg = QSM_REG_IDENTITY;
}

void qsm_rts_params_default(qsm_rts_params* p) {
    if (!p) return;  // src/inversion/rts.rs:41-52
    p->delta = 0.15;
    p->mu = 1e5;
    p->rho = 10.0;
    p->tol = 1e-2;
    p->max_iter = 20;
    p->lsmr_iter = 4;
}

void qsm_sharp_params_default(qsm_sharp_params* p) {
    if (!p) return;  // src/bgremove/sharp.rs:38-45
    p->threshold = 0.05;
    p->radius = 6.0;
}

int qsm_tkd(const double* local_field, const uint8_t* mask, const qsm_grid* grid, const double bdir[3],
            const qsm_tkd_params* params, double* chi_out) {
    g_err.clear();
    if (!params || !(params->threshold > 0)) return fail(QSM_EPARAM, "TKD threshold must be > 0");
    return filter_host(0, params->threshold, local_field, mask, grid, bdir, chi_out);
}

int qsm_tsvd(const double* local_field, const uint8_t* mask, const qsm_grid* grid, const double bdir[3],
             const qsm_tkd_params* params, double* chi_out) {
    g_err.clear();
    if (!params || std::isnan(params->threshold)) return fail(QSM_EPARAM, "TSVD threshold is NaN");
    return filter_host(1, params->threshold, local_field, mask, grid, bdir, chi_out);
}

int qsm_tikhonov(const double* local_field, const uint8_t* mask, const qsm_grid* grid,
                 const double bdir[3], const qsm_tikhonov_params* params, double* chi_out) {
    g_err.clear();
    if (!params || params->reg < QSM_REG_IDENTITY || params->reg > QSM_REG_LAPLACIAN)
        return fail(QSM_EPARAM, "bad Tikhonov parameters");
    return filter_host(2 + (int)params->reg, params->lambda, local_field, mask, grid, bdir, chi_out);
}

int qsm_rts(const double* local_field, const uint8_t* mask, const qsm_grid* grid, const double bdir[3],
            const qsm_rts_params* params, qsm_progress_fn progress, void* user, double* chi_out) {
    g_err.clear();
    if (!local_field || !mask || !grid || !bdir || !params || !chi_out)
        return fail(QSM_EPARAM, "null argument");
    int rc = validate_grid(grid);
    if (rc) return rc;
    const size_t N = grid->nx * grid->ny * grid->nz;
    HostVolume hv;
    qsm_tv_batch* B = nullptr;
    auto done = [&](int code) {
        if (B) batch_free(B);
        host_volume_free(hv);
        return code;
    };
    if ((rc = host_volume_upload(hv, local_field, mask, N))) return done(rc);
    const qsm_tv_volume vol = host_volume(grid, bdir);
    if ((rc = tv_batch_create_impl(&vol, 1, nullptr, nullptr, &B, params, &hv))) return done(rc);
    B->graph_state = -1;  // run once: capturing the graphs costs more than they save
    B->host_out = chi_out;
    B->host_bytes = N * sizeof(double);
    if ((rc = tv_batch_run_impl(B, progress, user))) return done(rc);
    if ((rc = host_volume_download(hv, chi_out, N))) return done(rc);
    return done(QSM_OK);
}

int qsm_rts_batch_create(const qsm_tv_volume* vols, size_t n_vols, const qsm_rts_params* params,
                         void* stream, qsm_tv_batch** out) {
    g_err.clear();
    if (!params) return fail(QSM_EPARAM, "null argument");
    return tv_batch_create_impl(vols, n_vols, nullptr, stream, out, params);
}

int qsm_sharp(const double* field, const uint8_t* mask, const qsm_grid* grid,
              const qsm_sharp_params* params, double* local_out, uint8_t* mask_out) {
    g_err.clear();
    if (!params) return fail(QSM_EPARAM, "null argument");
    const double r = params->radius;
    return vsharp_host(field, mask, grid, &r, 1, params->threshold, nullptr, nullptr, local_out,
                       mask_out);
}

void qsm_inversion_config_default(qsm_inversion_config* c) {
    if (!c) return;  // src/pipeline/config.rs:248-264
    c->algorithm = QSM_INV_RTS;
    qsm_tkd_params_default(&c->tkd);
    qsm_tkd_params_default(&c->tsvd);
    qsm_tikhonov_params_default(&c->tikhonov);
    qsm_tv_params_default(&c->tv);
    qsm_rts_params_default(&c->rts);
    qsm_nltv_params_default(&c->nltv);
}

// run_dipole_inversion, src/pipeline/inversion.rs:28-114, for the arms with
// a GPU backend here (Tkd, Tsvd, Tikhonov, Tv, Rts, Nltv).
int qsm_run_dipole_inversion_cfg(const double* local_field_ppm, size_t field_len, const uint8_t* mask,
                                 size_t mask_len, const qsm_scan_metadata* md,
                                 const qsm_inversion_config* cfg, qsm_progress_fn progress, void* user,
                                 double* chi_out) {
    g_err.clear();
    if (!md || !cfg) return fail(QSM_EPARAM, "metadata or config is null");
    const size_t n = md->nx * md->ny * md->nz;
    if (field_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, field_len);
    if (mask_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, mask_len);
    qsm_grid g{md->nx, md->ny, md->nz, md->vsx, md->vsy, md->vsz};
    const double* b = md->b0_direction;
    switch (cfg->algorithm) {
        case QSM_INV_TKD: return qsm_tkd(local_field_ppm, mask, &g, b, &cfg->tkd, chi_out);
        case QSM_INV_TSVD: return qsm_tsvd(local_field_ppm, mask, &g, b, &cfg->tsvd, chi_out);
        case QSM_INV_TIKHONOV: return qsm_tikhonov(local_field_ppm, mask, &g, b, &cfg->tikhonov, chi_out);
        case QSM_INV_TV: return qsm_tv_admm(local_field_ppm, mask, &g, b, &cfg->tv, progress, user, chi_out);
        case QSM_INV_RTS: return qsm_rts(local_field_ppm, mask, &g, b, &cfg->rts, progress, user, chi_out);
        case QSM_INV_NLTV: return qsm_nltv(local_field_ppm, mask, &g, b, &cfg->nltv, progress, user, chi_out);
        case QSM_INV_TGV:
        case QSM_INV_QSMART:
            return fail(QSM_ECONFIG, "invalid config: %s should use run_tgv or run_qsmart",
                        cfg->algorithm == QSM_INV_TGV ? "Tgv" : "Qsmart");
        default:
            return fail(QSM_ECONFIG, "invalid config: algorithm %d has no GPU backend here",
                        (int)cfg->algorithm);
    }
}

int qsm_vsharp_batch_create(const qsm_vsharp_volume* vols, size_t n_vols, const double* radii,
                            size_t n_radii, double threshold, void* stream, qsm_vsharp_batch** out) {
    g_err.clear();
    return vs_create_impl(vols, n_vols, radii, n_radii, threshold, stream, out);
}

int qsm_vsharp_batch_run(qsm_vsharp_batch* batch, qsm_progress_fn progress, void* user) {
    g_err.clear();
    return vs_run_impl(batch, progress, user);
}

void qsm_vsharp_batch_destroy(qsm_vsharp_batch* batch) { vs_free(batch); }

int qsm_vsharp_with_radii(const double* field, const uint8_t* mask, const qsm_grid* grid,
                          const double* radii, size_t n_radii, double threshold,
                          qsm_progress_fn progress, void* user, double* local_out,
                          uint8_t* mask_out) {
    g_err.clear();
    return vsharp_host(field, mask, grid, radii, n_radii, threshold, progress, user, local_out,
                       mask_out);
}

int qsm_vsharp(const double* field, const uint8_t* mask, const qsm_grid* grid,
               const qsm_vsharp_params* params, qsm_progress_fn progress, void* user,
               double* local_out, uint8_t* mask_out) {
    g_err.clear();
    if (!params) return fail(QSM_EPARAM, "params is null");
    std::vector<double> radii;
    int rc = vsharp_radii(params, radii);
    if (rc) return rc;
    return vsharp_host(field, mask, grid, radii.data(), radii.size(), params->threshold, progress,
                       user, local_out, mask_out);
}

int qsm_run_bg_removal(const double* field_ppm, size_t field_len, const uint8_t* mask,
                       size_t mask_len, const qsm_scan_metadata* md,
                       qsm_bg_removal_algorithm algorithm, const qsm_vsharp_params* vsharp_params,
                       qsm_progress_fn progress, void* user, double* local_out, uint8_t* mask_out) {
    g_err.clear();
    if (!md) return fail(QSM_EPARAM, "metadata is null");
    const size_t n = md->nx * md->ny * md->nz;
    // src/pipeline/bg_removal.rs:30-35
    if (field_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, field_len);
    if (mask_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, mask_len);
    qsm_bg_removal_config cfg;
    qsm_bg_removal_config_default(&cfg);
    cfg.algorithm = algorithm;
    if (vsharp_params) cfg.vsharp = *vsharp_params;
    return qsm_run_bg_removal_cfg(field_ppm, field_len, mask, mask_len, md, &cfg, progress, user,
                                  local_out, mask_out);
}

void qsm_bg_removal_config_default(qsm_bg_removal_config* c) {
    if (!c) return;  // src/pipeline/config.rs:215-229
    c->algorithm = QSM_BG_VSHARP;
    qsm_vsharp_params_default(&c->vsharp);
    qsm_sharp_params_default(&c->sharp);
}

// run_bg_removal, src/pipeline/bg_removal.rs:20-92, for the Vsharp and Sharp
// arms.
int qsm_run_bg_removal_cfg(const double* field_ppm, size_t field_len, const uint8_t* mask,
                           size_t mask_len, const qsm_scan_metadata* md,
                           const qsm_bg_removal_config* cfg, qsm_progress_fn progress, void* user,
                           double* local_out, uint8_t* mask_out) {
    g_err.clear();
    if (!md || !cfg) return fail(QSM_EPARAM, "metadata or config is null");
    const size_t n = md->nx * md->ny * md->nz;
    if (field_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, field_len);
    if (mask_len != n) return fail(QSM_EDIM, "dimension mismatch: expected %zu, got %zu", n, mask_len);
    qsm_grid g{md->nx, md->ny, md->nz, md->vsx, md->vsy, md->vsz};
    switch (cfg->algorithm) {
        case QSM_BG_VSHARP:
            return qsm_vsharp(field_ppm, mask, &g, &cfg->vsharp, progress, user, local_out, mask_out);
        case QSM_BG_SHARP:
            return qsm_sharp(field_ppm, mask, &g, &cfg->sharp, local_out, mask_out);
        default:
            return fail(QSM_ECONFIG, "invalid config: algorithm %d has no GPU backend here",
                        (int)cfg->algorithm);
    }
}

// Best rate of `reps` timed launches of `launch` moving `bytes` (GB/s),
// after one untimed launch.
extern "C++" {
template <class F>
static hipError_t best_rate(int reps, double bytes, F launch, double& best) {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) { launch(); e = hipGetLastError(); }
    best = 0.0;
    for (int r = 0; r < reps && e == hipSuccess; ++r) {
        float ms = 0.f;
        if ((e = hipEventRecord(e0, nullptr)) != hipSuccess) break;
        launch();
        if ((e = hipGetLastError()) != hipSuccess) break;
        if ((e = hipEventRecord(e1, nullptr)) != hipSuccess) break;
        if ((e = hipEventSynchronize(e1)) != hipSuccess) break;
        if ((e = hipEventElapsedTime(&ms, e0, e1)) != hipSuccess) break;
        const double g = bytes / (ms * 1e-3) / 1e9;
        if (g > best) best = g;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return e;
}
}  // extern "C++"

// Device-to-device copy rate of a plain one-element-per-thread kernel over
// `bytes` (read + write counted), best of `reps` timed launches.
int qsm_hbm_copy_probe(size_t bytes, int reps, double* gbps) {
    g_err.clear();
    if (!gbps || bytes < 16 || reps < 1) return fail(QSM_EPARAM, "bad probe arguments");
    const size_t n = bytes / sizeof(float2);
    float2 *a = nullptr, *b = nullptr;
    int rc;
    if ((rc = dev_alloc(&a, n)) || (rc = dev_alloc(&b, n))) {
        workspace_free(a);
        return rc;
    }
    launch_fill_zero(nullptr, reinterpret_cast<float*>(a), 2 * n);
    double best = 0.0;
    const hipError_t e = best_rate(reps, 2.0 * (double)n * sizeof(float2),
                                   [&] { launch_copy_probe(nullptr, a, b, n); }, best);
    workspace_free(a);
    workspace_free(b);
    if (e != hipSuccess) return fail(QSM_EHIP, "copy probe: %s", hipGetErrorString(e));
    *gbps = best;
    return QSM_OK;
}

// Rate of a pass shape: `reads` arrays of n floats read and `writes` arrays
// written element by element (1..4 each), all bytes counted.
int qsm_hbm_stream_probe(size_t n, int reads, int writes, int reps, double* gbps) {
    g_err.clear();
    if (!gbps || n < 4096 || reps < 1 || reads < 1 || reads > 4 || writes < 1 || writes > 4)
        return fail(QSM_EPARAM, "bad probe arguments");
    float *in = nullptr, *out = nullptr;
    int rc;
    if ((rc = dev_alloc(&in, n * reads)) || (rc = dev_alloc(&out, n * writes))) {
        workspace_free(in);
        return rc;
    }
    launch_fill_zero(nullptr, in, n * reads);
    double best = 0.0;
    const hipError_t e = best_rate(reps, 4.0 * (double)n * (reads + writes),
                                   [&] { launch_stream_probe(nullptr, reads, writes, in, out, n); }, best);
    workspace_free(in);
    workspace_free(out);
    if (e != hipSuccess) return fail(QSM_EHIP, "stream probe: %s", hipGetErrorString(e));
    *gbps = best;
    return QSM_OK;
}

int qsm_device_alloc(size_t bytes, void** out) {
    g_err.clear();
    if (!out) return fail(QSM_EPARAM, "null output pointer");
    *out = nullptr;
    const hipError_t e = with_trim([&] { return hipMalloc(out, bytes ? bytes : 1); });
    if (e != hipSuccess) {
        *out = nullptr;
        return fail(e == hipErrorOutOfMemory ? QSM_ENOMEM : QSM_EHIP, "hipMalloc(%zu bytes): %s", bytes,
                    hipGetErrorString(e));
    }
    return QSM_OK;
}

int qsm_device_free(void* ptr) {
    g_err.clear();
    if (ptr) QSM_HIP(hipFree(ptr));
    return QSM_OK;
}

int qsm_memcpy_htod(void* dst, const void* src, size_t bytes) {
    g_err.clear();
    if ((!dst || !src) && bytes) return fail(QSM_EPARAM, "null pointer");
    if (bytes) QSM_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return QSM_OK;
}

int qsm_memcpy_dtoh(void* dst, const void* src, size_t bytes) {
    g_err.clear();
    if ((!dst || !src) && bytes) return fail(QSM_EPARAM, "null pointer");
    if (bytes) QSM_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return QSM_OK;
}

int qsm_memcpy_dtod(void* dst, const void* src, size_t bytes) {
    g_err.clear();
    if ((!dst || !src) && bytes) return fail(QSM_EPARAM, "null pointer");
    if (bytes) QSM_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
    return QSM_OK;
}

int qsm_device_synchronize(void) {
    g_err.clear();
    QSM_HIP(hipDeviceSynchronize());
    return QSM_OK;
}

void qsm_release_cached_memory(void) { workspace_trim(); }

}  // extern "C"
