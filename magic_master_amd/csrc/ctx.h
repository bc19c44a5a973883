// Internal declarations shared by the C ABI (capi.hip) and the batched
// driver (batch.hip): the per-grid context, timing spans and host helpers.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../include/magic_hip.h"
#include "bc_src.h"
#include "magic_dev.h"
#include "parts.h"

using namespace magic;

#define HIPCHECK(x)                                                                   \
    do {                                                                              \
        hipError_t e_ = (x);                                                          \
        if (e_ != hipSuccess) {                                                       \
            fprintf(stderr, "magic_hip: %s failed: %s (%s:%d)\n", #x,                 \
                    hipGetErrorString(e_), __FILE__, __LINE__);                       \
            return MAGIC_EHIP;                                                        \
        }                                                                             \
    } while (0)

#define TRY(x)                        \
    do {                              \
        int s_ = (x);                 \
        if (s_ != MAGIC_OK) return s_; \
    } while (0)

// pinned host words of a context and where the global sums land in them
constexpr int HSCAL_WORDS = 32, HSCAL_SUMS = 16;

enum { AX_RHO = 0, AX_MX, AX_MY, AX_MZ, AX_E, AX_NU, AX_KAP, AX_VG, AX_R, AX_GAM, NAUXP };
enum { TC_SWX = 0, TC_SWY, TC_SWZ, TC_BC, TC_SRC, TC_OTHER, NTC };

struct TimedSpan {
    int cls;               // NTC: a launch of several sweep directions, shared by them
    hipEvent_t a, b;
    int nlaunch;
    float share[3];        // of each direction (cls = NTC)
};

// A slab of a grid swept on its own: its cells (Fortran i) i0 .. i1-1 of all
// rows and layers, and the blocks that hold increments of theirs: chunks of the
// x-sweep, tiles of the others, lo .. hi-1 of each direction.
struct Slab {
    int i0, i1;
    int lo[3], hi[3];
};

struct magic_ctx {
    int form = MAGIC_FORM_FP64;
    int mx, my, mz, meqn, mbc, maux;
    double xlower, ylower, zlower, dx, dy, dz;
    Dims d;
    long long P;
    hipStream_t stream = nullptr;
    double *q = nullptr, *qold = nullptr, *aux = nullptr, *zratio = nullptr;
    double *stage = nullptr, *u = nullptr, *qt = nullptr, *ut = nullptr;
    // FP32 perturbation form: state planes and scratch, background columns
    // (float: nu, kappa; FP64: rho, E, gamma, R, aux17, z residual)
    float *q32 = nullptr, *qold32 = nullptr, *u32 = nullptr, *qt32 = nullptr, *ut32 = nullptr;
    float *col32 = nullptr;
    double *bg64 = nullptr;
    Zr32 zr32;
    // FP64 form: when every aux slot the source pass reads is constant on
    // each layer (bitwise), those slots also live as columns (index k+mbc-1,
    // AX_ order) and the source pass reads the columns instead of the planes
    double *col64 = nullptr;
    bool aux_layered = false;
    bool own_stream = true;   // false when a batch lends its stream
    // The sweeps' increment blocks (SweepParts) of one step, of the whole grid
    // or, where the device has no room for that, of one of its slabs at a time.
    // Allocated on first use.
    void *parts = nullptr;
    size_t parts_bytes = 0;
    bool parts_stage = false;         // they lie in stage: there is no room beside it
    size_t parts_room = ~size_t(0);   // bytes the caller allows them
    std::vector<Slab> slabs;          // one: the whole grid
    // Inside magic_claw3 the increments of a step are left to the source
    // pass's conversion (pending), which adds them on its way
    bool pending_parts = false;
    StepParts<double> parts64;   // the last sweeps' increments, by form
    StepParts<float> parts32;
    // Asynchronous snapshots (magic_snapshot_begin): the conversion into
    // stage runs on the context's stream, the copy out of stage on cstream
    // (created on first use), so that later work on the stream need not
    // wait for the copy.  snap_done marks the last such copy; every other
    // user of stage waits for it first (stage_ready).
    hipStream_t cstream = nullptr;
    hipEvent_t snap_conv = nullptr, snap_done = nullptr;
    bool snap_pending = false;
    unsigned long long *dscal = nullptr;   // [0] cfl bits, [1..] status ints
    int shape[3] = {0, 0, 0};              // tile shape of the x-, y- and z-sweeps
    // The sweep kernel's operands (set up on the first tiled sweep): an
    // argument block per direction (written by a kernel at the start of each
    // step3 or of each tuner round), run flags all pointing at a device 1, and
    // the workgroups' blocks, slab by slab and direction by direction (those of
    // slab s and direction d at [item_off[3 s + d], item_off[3 s + d + 1]))
    void *largs = nullptr;
    const int **lrun = nullptr;
    int *lone = nullptr;
    int4 *items = nullptr;
    std::vector<int> item_off;
    int item_shape[3] = {-1, -1, -1};      // the shapes the items were laid out for
    GridGate gate;                         // of the kernels launched now (claw3's source pass)
    unsigned long long *hscal = nullptr;   // pinned host words: [0, 8) mirror dscal, [HSCAL_SUMS, +10) global sums
    void *sums_d = nullptr;                // global sums: partials and results (first magic_global_sums)
    magic_params prm;
    bool have_params = false, have_aux = false;
    double aux11_top = 0.0, aux12_top = 0.0;
    int errloc[4] = {0, 0, 0, 0};
    bool timing = false;
    double ms[NTC] = {0};
    long long launches[NTC] = {0};
    std::vector<TimedSpan> pending;
    std::vector<hipEvent_t> pool;
};

// ------------------------------------------------------------ timing -----
static inline hipEvent_t ev_get(magic_ctx *c)
{
    hipEvent_t e;
    if (!c->pool.empty()) {
        e = c->pool.back();
        c->pool.pop_back();
    } else if (hipEventCreate(&e) != hipSuccess) {
        return nullptr;
    }
    return e;
}

struct Span {
    magic_ctx *c;
    int cls, n;
    hipStream_t s;
    hipEvent_t a = nullptr;
    float share[3] = {0.f, 0.f, 0.f};
    Span(magic_ctx *c_, int cls_, int n_, hipStream_t s_ = nullptr) : c(c_), cls(cls_), n(n_), s(s_ ? s_ : c_->stream)
    {
        if (c->timing && (a = ev_get(c))) hipEventRecord(a, s);
    }
    ~Span()
    {
        if (!c->timing) {
            return;
        }
        hipEvent_t b = ev_get(c);
        if (a && b) {
            hipEventRecord(b, s);
            c->pending.push_back({cls, a, b, n, {share[0], share[1], share[2]}});
        }
    }
};

static inline void drain_timing(magic_ctx *c)
{
    for (auto &s : c->pending) {
        float ms = 0.f;
        if (hipEventSynchronize(s.b) == hipSuccess && hipEventElapsedTime(&ms, s.a, s.b) == hipSuccess) {
            if (s.cls < NTC) {
                c->ms[s.cls] += ms;
                c->launches[s.cls] += s.nlaunch;
            } else {
                for (int d = 0; d < 3; d++)
                    if (s.share[d] > 0.f) {
                        c->ms[TC_SWX + d] += ms * s.share[d];
                        c->launches[TC_SWX + d] += s.nlaunch;
                    }
            }
        }
        c->pool.push_back(s.a);
        c->pool.push_back(s.b);
    }
    c->pending.clear();
}

// ---------------------------------------------------------- helpers ------
static inline unsigned blocks(long long n, int b) { return (unsigned)((n + b - 1) / b); }

static inline int launch_check() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        fprintf(stderr, "magic_hip: kernel launch failed: %s\n", hipGetErrorString(e));
        return MAGIC_EHIP;
    }
    return MAGIC_OK;
}

static inline int ntracer(const magic_ctx *c) { return c->meqn - 5; }

// Launch shape of the per-cell kernels (INTERIOR_IJK, PADDED_IJK): 64 cells
// along x by 4 rows along y per workgroup, one layer per grid z index.
static inline dim3 cell_block() { return dim3(64, 4, 1); }
static inline dim3 interior_grid(const Dims &d) { return dim3(blocks(d.mx, 64), blocks(d.my, 4), d.mz); }
static inline dim3 slab_cells(const Dims &d, const Slab &s) { return dim3(blocks(s.i1 - s.i0, 64), blocks(d.NY, 4), d.NZ); }
static inline dim3 padded_cells(const Dims &d) { return dim3(blocks(d.NX, 64), blocks(d.NY, 4), d.NZ); }
// Layers per workgroup of the diffusion kernels, cols workgroups side by side.
// Each workgroup's layers run one after the other, so many short workgroups
// hide the latency better, but each loads (cross terms) or forms (directional
// passes) two layers beside its own: about most workgroups, at least 4 layers
// each where that still makes 512 of them (12 x 10 x 8: the cross terms 9.0 ->
// 5.0 us with one layer each).
static inline int layers_kb(const Dims &d, long long cols, long long most)
{
    auto kb_for = [&](long long groups) {
        const long long chunks = (groups + cols - 1) / cols;
        return (int)((d.mz + chunks - 1) / chunks);
    };
    return std::max(kb_for(most), std::min(4, kb_for(512)));
}
static inline dim3 diff_cols(const Dims &d) { return dim3(blocks(d.mx, 64), blocks(d.my, 4)); }
static inline dim3 passes_cols(const Dims &d) { return dim3(blocks(d.mx, 64), blocks(d.my, 4 * DIFF_ROWS)); }
static inline int diff_kb(const Dims &d) { return layers_kb(d, (long long)diff_cols(d).x * diff_cols(d).y, 8192); }
// (the directional passes of four components run side by side in one launch)
static inline int passes_kb(const Dims &d)
{
    return layers_kb(d, 4ll * passes_cols(d).x * passes_cols(d).y, 4096);
}
static inline dim3 diff_grid(const Dims &d) { return dim3(diff_cols(d).x, diff_cols(d).y, blocks(d.mz, diff_kb(d))); }
static inline dim3 passes_grid(const Dims &d, int comps)
{
    return dim3(passes_cols(d).x, passes_cols(d).y, comps * blocks(d.mz, passes_kb(d)));
}

// every tracer count of meqn 5 .. 10 (rpt3euX.f:134-138 splits tracers 6 .. meqn)
static inline bool sweep_supported(int ntr) { return ntr >= 0 && ntr <= 5; }

// ------------------------------------------------------- tile shapes ----
// The tiled sweep kernel of shape sh (0 .. TILE_NSHAPE-1), launched for one
// grid and for a batch of grids alike.
template <typename T, bool PERT, int NTR>
static inline const void *tile_fn_n(int sh)
{
    switch (sh) {
    case 0: return reinterpret_cast<const void *>(&tile_sweep<T, PERT, NTR, 0>);
    case 1: return reinterpret_cast<const void *>(&tile_sweep<T, PERT, NTR, 1>);
    case 2: return reinterpret_cast<const void *>(&tile_sweep<T, PERT, NTR, 2>);
    case 3: return reinterpret_cast<const void *>(&tile_sweep<T, PERT, NTR, 3>);
    default: return nullptr;
    }
}
static_assert(TILE_NSHAPE == 4, "tile_fn_n lists every shape");
template <typename T, bool PERT>
static inline const void *tile_fn(int ntr, int sh)
{
    switch (ntr) {
    case 0: return tile_fn_n<T, PERT, 0>(sh);
    case 1: return tile_fn_n<T, PERT, 1>(sh);
    case 2: return tile_fn_n<T, PERT, 2>(sh);
    case 3: return tile_fn_n<T, PERT, 3>(sh);
    case 4: return tile_fn_n<T, PERT, 4>(sh);
    case 5: return tile_fn_n<T, PERT, 5>(sh);
    default: return nullptr;
    }
}

// log2 of the planes per segment of a grid's sweeps.  Longer segments write
// and read fewer edge planes (L + 2 for L) and start less often; shorter ones
// give more workgroups.  The estimate, in planes of work: a segment costs its
// planes and 1.5 for its start and its two extra planes, at_once workgroups run
// at a time, and the last ones leave the chip idle for 0.65 of a segment (less
// where hardly any are left after the first).  It depends on the grid alone
// (not on the device or on a batch's other grids), since the sums' grouping,
// and so the last bits, depend on it.  Measured, ms per step with 4, 8, 16, 32 planes:
// 250 x 200 x 300 FP64 6.13, 5.82, 5.62, 5.54 (takes 32); 128 x 100 x 150 with
// five tracers 1.87, 1.77, 1.74, 1.72 (16); 181 x 160 x 243 FP32 2.22, 2.08, 2.06,
// 2.09 (16); 64 x 64 x 96 FP32 0.232, 0.222, 0.216, 0.340 (16); 64 x 64 x 48
// FP64 0.185, 0.175, 0.259, 0.295 (8); 110 x 90 x 140 FP64 0.701, 0.684, 0.672,
// 0.738 (8); 72 x 66 x 104 FP32 0.289, 0.282, 0.296, 0.348 (8).
static inline int segment_lg(const Dims &d, double at_once)
{
    auto cols = [](int n, int a) { return (long long)((a + 2 + 15) / 16) * ((n + 1 + 13) / 14); };
    const long long cxy = cols(d.mx, d.my) + cols(d.my, d.mx), cz = cols(d.mz, d.mx);
    int best = 0;
    double fbest = 0.0;
    for (int lg = 0; lg <= 5; lg++) {
        const int L = 1 << lg;
        auto segs = [&](int nB) { return (nB + 2 + L - 1) >> lg; };
        const double rounds = (double)(cxy * segs(d.mz) + cz * segs(d.my)) / at_once;
        const double work = (cxy * (d.mz + 2 + 1.5 * segs(d.mz)) + cz * (d.my + 2 + 1.5 * segs(d.my))) / at_once;
        const double f = std::max(work, L + 1.5) + 0.65 * L * std::min(1.0, std::max(0.0, 10.0 * (rounds - 1.0)));
        if (lg == 0 || f < fbest) {
            best = lg;
            fbest = f;
        }
    }
    return best;
}

// The part of direction dir's argument block that the grid fixes: planes of
// the components, strides and the layout of its blocks.  The tile axis is g
// for the x- and z-sweeps (lib/step3.f:121-280 g = y, h = z; 459-621 g = x,
// h = y) and x = h for the y-sweep (289-450 g = z, h = x), so that the y- and
// z-sweeps tile along rows of x.
template <typename T>
static inline void sweep_geometry(const magic_ctx *c, int dir, int sh, SweepArgsT<T> &a, SweepParts<T> &p)
{
    const Dims &d = c->d;
    const long long NXY = (long long)d.NX * d.NY;
    static const int comp[3][5] = {{0, 1, 2, 3, 4}, {0, 2, 3, 1, 4}, {0, 3, 1, 2, 4}};
    for (int m = 0; m < 5; m++) a.comp[m] = comp[dir][m];
    for (int m = 5; m < c->meqn; m++) a.comp[m] = m;
    a.P = c->P;
    a.mbc = c->mbc;
    a.n = dir == 0 ? c->mx : dir == 1 ? c->my : c->mz;
    a.nA = dir == 0 ? c->my : c->mx;
    a.nB = dir == 2 ? c->my : c->mz;
    a.sN = dir == 0 ? 1 : dir == 1 ? d.NX : NXY;
    a.sA = dir == 0 ? d.NX : 1;
    a.sB = dir == 2 ? d.NX : NXY;
    a.a_is_g = dir != 1;
    for (int m = 0; m < 10; m++)
        a.cofs[m] = d.P * (m == 2 ? a.comp[a.a_is_g ? 2 : 3] : m == 3 ? a.comp[a.a_is_g ? 3 : 2] : m < c->meqn ? a.comp[m] : 0);
    a.gravity = dir == 2;
    a.sweep = dir + 1;
    memset(&p, 0, sizeof(p));
    p.n = a.n; p.nA = a.nA; p.nB = a.nB;
    p.lgTA = tile_lgta(sh);
    // two workgroups per compute unit.  A third (FP32), or a second with four
    // tracers or more in FP64, runs beside the others but makes them slower: with
    // segments chosen for 768 at once 40 x 36 x 60 FP32 takes 0.139 ms instead of
    // 0.119, and for 512 97 x 83 x 121 with five tracers 0.784 instead of 0.706.
    p.lgL = segment_lg(d, sizeof(T) == 8 && c->meqn >= 9 ? 256.0 : 512.0);
    p.CI = tile_ci(sh);
    p.iCI = (unsigned)(((1ull << 32) + p.CI - 1) / p.CI);
    p.nt = (a.nA + 2 + tile_ta(sh) - 1) / tile_ta(sh);
    p.nk = (a.n + 1 + p.CI - 1) / p.CI;
    p.ns = (a.nB + 2 + (1 << p.lgL) - 1) >> p.lgL;
    p.sT = dir == 0 ? p.nk : 1;
    p.sK = dir == 0 ? 1 : p.nt;
    p.sS = p.nk * p.nt;
    a.lgL = p.lgL; a.sT = p.sT; a.sK = p.sK; a.sS = p.sS;
}
template <typename T>
static inline void sweep_factors(const magic_ctx *c, int dir, double dt, SweepArgsT<T> &a)
{
    const double x = dt / c->dx, y = dt / c->dy, z = dt / c->dz;
    a.dtdn = dir == 0 ? x : dir == 1 ? y : z;
    a.fg = dir == 0 ? y : dir == 1 ? z : x;
    a.fh = dir == 0 ? z : dir == 1 ? x : y;
}
// Elements of one block
template <typename T>
static inline long long block_size(const SweepParts<T> &p, int nc, int sh)
{
    return (long long)((1 << p.lgL) + 2) * nc * part_npos(sh);
}
// The blocks lo .. hi-1 along x of direction dir laid out from next on;
// returns the element behind them.
template <typename T>
static inline T *parts_layout(SweepArgsT<T> &a, SweepParts<T> &p, int dir, int lo, int hi, int nc, int sh, T *next)
{
    const int w = hi - lo;
    p.sT = dir == 0 ? w : 1;
    p.sK = dir == 0 ? 1 : w;
    p.sS = w * (dir == 0 ? p.nt : p.nk);
    const long long bs = block_size(p, nc, sh);
    a.parts = next - lo * bs;
    p.base = a.parts;
    a.sT = p.sT; a.sK = p.sK; a.sS = p.sS;
    return next + bs * p.sS * p.ns;
}
// the blocks lo .. hi-1 along x of one direction, as they lie in the part buffer
template <typename T>
static inline void push_items(std::vector<int4> &items, const SweepParts<T> &p, int dir, int lo, int hi, int arg)
{
    const int kl = dir == 0 ? lo : 0, kh = dir == 0 ? hi : p.nk, tl = dir == 0 ? 0 : lo, th = dir == 0 ? p.nt : hi;
    for (int s = 0; s < p.ns; s++)
        for (int k = kl; k < kh; k++)
            for (int t = tl; t < th; t++) items.push_back(make_int4(arg, t, k, s));
}

// The blocks along x that hold entries of the cells i0 .. i1-1, as add_parts
// (parts.h) looks them up: a cell's own block and, next to an edge, the
// neighbouring one; cells without entries look at the nearest column's.
template <typename T>
static inline void slab_blocks(const SweepParts<T> &p, int dir, int i0, int i1, int &lo, int &hi)
{
    auto clamp = [](int x, int a, int b) { return std::min(std::max(x, a), b); };
    if (dir == 0) {
        const int x = clamp(i1 - 2, 0, p.n - 1);
        lo = clamp(i0 - 1, 0, p.n - 1) / p.CI;
        hi = x / p.CI + (x % p.CI == p.CI - 1 ? 2 : 1);
    } else {
        const int TA = 1 << p.lgTA;
        const int x = clamp(i0, -1, p.nA + 2), y = clamp(i1 - 1, -1, p.nA + 2);
        lo = x < 0 ? 0 : x / TA - (x >= 1 && x % TA == 0 ? 1 : 0);
        hi = y < 0 ? 1 : std::min(p.nt, y / TA + (y % TA == TA - 1 ? 2 : 1));
    }
}

// Slabs of a grid's sweeps in shapes sh.  A slab sweeps every block that holds
// entries of its cells, so each cell's sum is whole and in its one order; slabs
// share the blocks at their borders, which are swept twice: 16 cells wide, about
// three times the work.
constexpr int SLAB_MIN = 16;
template <typename T>
struct Slabs {
    int mx, mbc;
    SweepParts<T> p[3];
    long long row[3];   // bytes of the blocks at one place along x
    Slabs(const magic_ctx *c, const int *sh) : mx(c->mx), mbc(c->mbc)
    {
        for (int dir = 0; dir < 3; dir++) {
            SweepArgsT<T> a;
            sweep_geometry(c, dir, sh[dir], a, p[dir]);
            row[dir] = block_size(p[dir], c->meqn, sh[dir]) * (dir == 0 ? p[dir].nt : p[dir].nk) * p[dir].ns * (long long)sizeof(T);
        }
    }
    // the slab of the cells x .. x+w-1 and what its increments take
    Slab at(int x, int w, size_t &bytes) const
    {
        Slab s;
        s.i0 = x == 0 ? 1 - mbc : x;
        s.i1 = x + w < mx + 2 ? x + w : mx + mbc + 1;
        bytes = 0;
        for (int dir = 0; dir < 3; dir++) {
            slab_blocks(p[dir], dir, s.i0, s.i1, s.lo[dir], s.hi[dir]);
            bytes += (size_t)(row[dir] * (s.hi[dir] - s.lo[dir]));
        }
        return s;
    }
    // slabs w cells wide; bytes: of the largest
    std::vector<Slab> cut(int w, size_t &bytes) const
    {
        std::vector<Slab> out;
        bytes = 0;
        for (int x = 0; x < mx + 2; x += w) {
            size_t n;
            out.push_back(at(x, w, n));
            bytes = std::max(bytes, n);
        }
        return out;
    }
    size_t whole() const   // what the increments of the whole grid take
    {
        size_t n;
        at(0, mx + 2, n);
        return n;
    }
    size_t least() const   // and those of the narrowest slabs
    {
        size_t n, most = 0;
        for (int x = 0; x < mx + 2; x += SLAB_MIN) {
            at(x, SLAB_MIN, n);
            most = std::max(most, n);
        }
        return most;
    }
    // the widest slabs whose increments take at most room bytes (least() at the least)
    std::vector<Slab> within(size_t room) const
    {
        size_t n;
        std::vector<Slab> s = cut(mx + 2, n);
        for (int w = (mx + 1) / SLAB_MIN * SLAB_MIN; n > room && w >= SLAB_MIN; w -= SLAB_MIN) s = cut(w, n);
        return s;
    }
};

// capi.hip
int tune_state(magic_ctx *c), tune_done(magic_ctx *c);
int failed_step(magic_ctx *c, const int *shape, double dt);
int stage_ready(magic_ctx *c);
static inline size_t stage_bytes(const magic_ctx *c) { return (size_t)c->P * c->meqn * sizeof(double); }

// Event pairs of the autotuners, one per (direction, shape).  The shapes
// are timed round-robin (every round times each candidate once), so that a
// drift of the clocks over the tuning run favours none of them.
struct TuneClock {
    hipEvent_t ev[3][TILE_NSHAPE][2] = {};
    float ms[3][TILE_NSHAPE] = {};
    bool ok = true;
    TuneClock()
    {
        for (auto &d : ev)
            for (auto &s : d)
                for (auto &e : s) ok = ok && hipEventCreate(&e) == hipSuccess;
    }
    ~TuneClock()
    {
        for (auto &d : ev)
            for (auto &s : d)
                for (auto &e : s)
                    if (e) hipEventDestroy(e);
    }
    int mark(int dir, int sh, int end, hipStream_t st)
    {
        return hipEventRecord(ev[dir][sh][end], st) == hipSuccess ? MAGIC_OK : MAGIC_EHIP;
    }
    // adds every pair of the round just recorded
    int add_round()
    {
        for (int d = 0; d < 3; d++)
            for (int s = 0; s < TILE_NSHAPE; s++) {
                float t = 0.f;
                if (hipEventSynchronize(ev[d][s][1]) != hipSuccess ||
                    hipEventElapsedTime(&t, ev[d][s][0], ev[d][s][1]) != hipSuccess)
                    return MAGIC_EHIP;
                ms[d][s] += t;
            }
        return MAGIC_OK;
    }
    // fastest shape per direction; mean ms per sweep over reps rounds
    void result(int reps, int best[3], float *ms_out) const
    {
        for (int d = 0; d < 3; d++) {
            best[d] = 0;
            for (int s = 1; s < TILE_NSHAPE; s++)
                if (ms[d][s] < ms[d][best[d]]) best[d] = s;
            if (ms_out)
                for (int s = 0; s < TILE_NSHAPE; s++) ms_out[d * TILE_NSHAPE + s] = ms[d][s] / (float)reps;
        }
    }
};

static inline bool shapes_valid(const int *sh)
{
    for (int k = 0; k < 3; k++)
        if (sh[k] < 0 || sh[k] >= TILE_NSHAPE) return false;
    return true;
}

// FP32 form's background columns (index kk = k + mbc - 1): float columns of
// the diffusivities, FP64 columns of everything its arithmetic reads
enum { C32_NU = 0, C32_KAP, NC32 };
enum { B64_RHO = 0, B64_E, B64_GAM, B64_R, B64_VG, B64_RES, NB64 };
static inline Col32 col32_of(const magic_ctx *c)
{
    const int NZ = c->d.NZ;
    return Col32{c->bg64 + B64_RHO * NZ, c->bg64 + B64_E * NZ, c->bg64 + B64_GAM * NZ, c->bg64 + B64_R * NZ};
}
