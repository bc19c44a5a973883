// Batched driver: many grids (scenarios) of one form (the FP32 perturbation
// form or the FP64 form) advanced together on one stream, with claw3's step
// control on the device (batch.h) and one attempted step of every scenario
// captured once as a HIP graph and replayed.
//
// One attempt:
//   prepare  (dt clip, per-grid sweep factors, source-pass substep counts)
//   bc3 (x, y, z faces), b4step3
//   per group of scenarios (as many as the increment buffer holds):
//     the sweeps    (one launch over the blocks of the group's grids)
//     decide        (accept / reject from the Courant number)
//     src3's conversion of the accepted scenarios, which adds the increments
//     to q and leaves the state before the step in the backup
//   the rest of src3 of accepted scenarios
//   finalize (next dt, step count, end of interval)
// The sweeps read q itself, which only an accepted step's conversion changes,
// so nothing is copied before a step or restored after a rejected one.
// Every launch covers all scenarios: the sweeps through lists of their blocks,
// the other kernels through block lists that lay the scenarios' own grids
// end to end (batch_ops.h), each scenario gated by its control block.  The
// number of launches per attempt does not depend on the number of
// scenarios; the source pass's substep loops run to the largest substep
// counts any scenario was started with (each scenario's own counts gate its
// part).  No host synchronisation inside an attempt; the host reads the
// control blocks back every few attempts to see whether all scenarios are
// done.
#include <algorithm>

#include "batch.h"
#include "batch_ops.h"
#include "ctx.h"

using namespace magic;

struct magic_batch {
    int n = 0;                           // slots in use (a removed scenario leaves an empty slot)
    int cap = 0;                         // slots the device arrays hold
    int meqn = 0, mbc = 0, maux = 0, form = 0;
    hipStream_t stream = nullptr;
    std::vector<magic_ctx *> sc;         // nullptr: empty slot
    std::vector<ScenCtl> ctl;            // host copy of the control blocks
    std::vector<int> mthbc;              // 6 per scenario
    std::vector<char> settled;           // a failed scenario's last step is in its q
    ScenCtl *ctl_d = nullptr;
    ScenCtl *ctl_pin = nullptr;          // pinned read-back buffer
    void *args_d = nullptr;              // SweepArgsT of the form, 3 per slot: one per direction
    const int **run_d = nullptr;         // per argument block: &ctl_d[s].run
    int4 *items_d = nullptr;
    // Groups of slots [lo, hi) whose increments the part buffer holds at
    // once; blocks of the group's direction d at items_d[off[d], off[d + 1]).
    // A grid too large for the buffer is a group for each of its slabs.
    struct Group {
        int lo, hi, off[4];
        int slab = -1, nslab = 0;        // of slot lo: which of how many (slab < 0: whole grids)
    };
    std::vector<Group> groups;
    std::vector<std::vector<Slab>> slabs;   // per slot; empty: swept whole
    std::vector<StepParts<double>> sp64; // per slot, by form: the increments of its sweeps
    std::vector<StepParts<float>> sp32;
    void *parts = nullptr;
    size_t parts_bytes = 0;
    magic_ctx *parts_of = nullptr;       // the scenario whose staging buffer it is: there is no room beside it
    size_t parts_room = 0;               // bytes the caller allows it (0: PARTS_BYTES)
    int shape[3] = {0, 0, 0};            // tile shape of the x-, y- and z-sweeps
    int *one_d = nullptr;                // a device 1: the run flag of every tile while tuning
    // boundary, copy and source-pass kernels (batch_ops.h)
    void *ops_d = nullptr;               // BatchOps of the form, one per slot
    int *loff_d = nullptr;               // NLG block lists: cap + 1 offsets each
    int4 *lgdim_d = nullptr;             //                  cap grid shapes each
    std::vector<int> loff;               // loff_d's host copy
    int ndtr_cap = 0, ndtrc_cap = 0;     // substep loops of the captured attempt
    int ncu = 0;                         // compute units
    int opgrid[NOP] = {0};               // persistent grid of each kernel class
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool dirty = true;                   // control blocks changed on the host
    bool graph_ok = false;
};

static StepParts<double> &slot_parts(magic_batch *b, int s, double) { return b->sp64[s]; }
static StepParts<float> &slot_parts(magic_batch *b, int s, float) { return b->sp32[s]; }
static bool fp32(const magic_batch *b) { return b->form == MAGIC_FORM_FP32P; }
static size_t elt(const magic_batch *b) { return fp32(b) ? sizeof(float) : sizeof(double); }
static double *state_q(const magic_ctx *c, double) { return c->q; }
static float *state_q(const magic_ctx *c, float) { return c->q32; }
static void *state_qold(const magic_ctx *c)
{
    return c->form == MAGIC_FORM_FP32P ? (void *)c->qold32 : (void *)c->qold;
}

// ------------------------------------------------------- control kernels --
template <typename T>
__global__ void k_batch_prepare(ScenCtl *ctl, int n, SweepArgsT<T> *args)
{
    const int s = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (s >= n) return;
    ScenCtl &c = ctl[s];
    c.accepted = 0;
    c.rejected = 0;
    c.run = c.active != 0 && c.status == 0;
    c.swept = c.run;
    if (!c.run) return;
    if (c.newstep) {                                   // claw3_mpi.f:741
        c.told = c.t;
        if (c.clip && c.told + c.dt > c.tend) c.dt = c.tend - c.told;
    }
    c.cfl_bits = 0ull;
    for (int e = 0; e < 6; e++) c.err[e] = 0;
    const double dt = c.dt;
    const double dtdx = dt / c.dx, dtdy = dt / c.dy, dtdz = dt / c.dz;
    SweepArgsT<T> &ax = args[s * 3], &ay = args[s * 3 + 1], &az = args[s * 3 + 2];
    ax.dtdn = dtdx; ax.fg = dtdy; ax.fh = dtdz;
    ay.dtdn = dtdy; ay.fg = dtdz; ay.fh = dtdx;
    az.dtdn = dtdz; az.fg = dtdx; az.fh = dtdy;
    // src3.f90:314-322
    const int ndtr = (int)ceil((dt * c.difmax / (c.dxyzmin2)) / 0.45);
    const double dtr = dt / ndtr;
    // ndtr = 0 (no viscosity at the top): no substep runs (src3.f90:341)
    const int ndtrc = ndtr > 0 ? (int)ceil((dtr * c.kapmax / (c.dxyzmin2)) / 0.45) : 0;
    const double dtrc = dtr / ndtrc;
    if (ndtr > c.ndtr_cap || ndtrc > c.ndtrc_cap) {   // beyond the captured substeps
        c.status = MAGIC_EUNSUPPORTED;
        c.run = 0;
        c.swept = 0;
        return;
    }
    c.ndtr = ndtr;
    c.ndtrc = ndtrc;
    c.dtr = dtr;
    c.dtrc = dtrc;
    // factors of the diffusion passes in the order the host form evaluates them
    const double fourthirds = 4.0 / 3.0;
    double dtdx2 = (dtr) / (c.dx * c.dx), dtdy2 = (dtr) / (c.dy * c.dy), dtdz2 = (dtr) / (c.dz * c.dz);
    const double dtr32 = dtr / 6.0;
    c.fac[FAC_CROSS + 0] = dtr32 / (c.dx * c.dy);
    c.fac[FAC_CROSS + 1] = dtr32 / (c.dx * c.dz);
    c.fac[FAC_CROSS + 2] = dtr32 / (c.dy * c.dz);
    for (int cc = 1; cc <= 3; cc++) {
        if (cc == 1) {
            dtdx2 = fourthirds * dtdx2;
        } else if (cc == 2) {
            dtdy2 = fourthirds * dtdy2;
            dtdx2 = dtdx2 / fourthirds;
        } else {
            dtdz2 = fourthirds * dtdz2;
            dtdy2 = dtdy2 / fourthirds;
        }
        c.fac[FAC_DIFF + 3 * (cc - 1) + 0] = dtdx2;
        c.fac[FAC_DIFF + 3 * (cc - 1) + 1] = dtdy2;
        c.fac[FAC_DIFF + 3 * (cc - 1) + 2] = dtdz2;
    }
    c.fac[FAC_COND + 0] = (dtrc) / (c.dx * c.dx);
    c.fac[FAC_COND + 1] = (dtrc) / (c.dy * c.dy);
    c.fac[FAC_COND + 2] = (dtrc) / (c.dz * c.dz);
    c.tgauss = exp(-.5 * ((c.told - c.tcenter) * (c.told - c.tcenter) / (c.twidth * c.twidth)));
}

// claw3_mpi.f:843-886: accept or reject the attempt
__global__ void k_batch_decide(ScenCtl *ctl, int n)
{
    const int s = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (s >= n) return;
    ScenCtl &c = ctl[s];
    if (!c.run) return;
    const double cfl = __longlong_as_double((long long)c.cfl_bits);
    c.cfl = cfl;
    c.attempts++;
    if (c.err[0] != 0) {
        c.status = c.err[0] == 1 ? MAGIC_ERHO : MAGIC_EA2;
        c.run = 0;
        c.active = 0;
        return;
    }
    if (cfl <= c.cflv1) {
        c.accepted = 1;
        c.t = c.told + c.dt;
        c.cflmax = c.cflmax > cfl ? c.cflmax : cfl;
    } else {
        c.rejected = 1;
        c.rejects++;
        c.t = c.told;
        c.dt = c.dtmax < c.dt * c.cflv2 / cfl ? c.dtmax : c.dt * c.cflv2 / cfl;
        c.newstep = 0;
    }
}

// claw3_mpi.f:910-927: next dt after an accepted step, end of the interval
__global__ void k_batch_finalize(ScenCtl *ctl, int n)
{
    const int s = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (s >= n) return;
    ScenCtl &c = ctl[s];
    if (!c.accepted) return;
    if (c.cfl == 0.0) c.dt = c.dtmax;
    else c.dt = c.dtmax < c.dt * c.cflv2 / c.cfl ? c.dtmax : c.dt * c.cflv2 / c.cfl;
    c.nsteps++;
    c.newstep = 1;
    if (c.t >= c.tend || c.nsteps >= c.maxsteps) c.active = 0;
}

// --------------------------------------------------------------- helpers --
// Substep counts of the source pass for any dt up to dtbound
// (src3.f90:314-322 at the largest dt).
static void src_caps(const magic_ctx *c, double dtbound, int *ndtr, int *ndtrc)
{
    double dmin = c->dx < c->dy ? c->dx : c->dy;
    dmin = dmin < c->dz ? dmin : c->dz;
    const double d2 = dmin * dmin;
    const double difmax = (4.0 / 3.0) * c->aux11_top;
    *ndtr = (int)std::ceil((dtbound * difmax / d2) / 0.45);
    if (*ndtr < 1) *ndtr = 1;
    // the conduction count is largest for the largest dtr, i.e. dt / 1
    *ndtrc = (int)std::ceil((dtbound * c->aux12_top / d2) / 0.45);
    if (*ndtrc < 1) *ndtrc = 1;
}

// the blocks of directions d0 .. d1-1 (of one shape) of a group's grids
template <typename T, bool PERT>
static int launch_dirs(magic_batch *b, const magic_batch::Group &g, int d0, int d1)
{
    const void *fn = tile_fn<T, PERT>(b->meqn - 5, b->shape[d0]);
    const int nblk = g.off[d1] - g.off[d0];
    if (!fn) return MAGIC_EARG;
    if (nblk <= 0) return MAGIC_OK;
    const SweepArgsT<T> *args = (const SweepArgsT<T> *)b->args_d;
    const int4 *items = b->items_d + g.off[d0];
    const int *const *run = b->run_d;
    void *kargs[] = {&args, &items, &run};
    HIPCHECK(hipLaunchKernel(fn, dim3((unsigned)nblk), dim3(256), kargs, 0, b->stream));
    return launch_check();
}

// Workgroup shape of the kernels that use block list lg
static dim3 list_block(int lg)
{
    switch (lg) {
    case LG_BC: case LG_BCUVW: case LG_CPY: return dim3(256);
    case LG_BCZ: return dim3(64);
    default: return cell_block();
    }
}

// The block list each kernel class walks
static int op_list(int op)
{
    static const int lg[NOP] = {LG_BC, LG_BCUVW, LG_BCZ, LG_CPY, LG_CPY, LG_PAD, LG_DIF, LG_DF4, LG_DF1, LG_INT, LG_INT};
    return lg[op];
}

// One launch of kernel class op over its block list (slots lo .. hi-1; all
// by default): a persistent grid of at most as many workgroups as fit on the
// chip at once
template <typename T>
static int launch_op(magic_batch *b, int op, GateSpec gs, int arg = 0, int lo = 0, int hi = -1)
{
    const int lg = op_list(op);
    if (hi < 0) hi = b->n;
    const int total = (int)(b->loff[(size_t)lg * (b->cap + 1) + hi] - b->loff[(size_t)lg * (b->cap + 1) + lo]);
    if (total <= 0) return MAGIC_OK;
    const void *fn = batch_op_fn<T>(op);
    if (!fn || b->opgrid[op] < 1) return MAGIC_EARG;
    const BatchOps<T> *ops = (const BatchOps<T> *)b->ops_d + lo;
    const int *off = b->loff_d + (size_t)lg * (b->cap + 1) + lo;
    const int4 *gd = b->lgdim_d + (size_t)lg * b->cap + lo;
    int n = hi - lo;
    void *kargs[] = {&ops, &off, &gd, &n, &gs, &arg};
    int grid = b->opgrid[op];
    // The conversion gathers from 18 or more places per cell.  Where the
    // increments (256 cells to a block, three directions) come from memory
    // and not from the 256 MB cache before it, fewer workgroups at once keep
    // to fewer pages: 8 FP32 grids of 200 x 200 x 300 take 2.56 ms with three
    // per compute unit, 2.75 with four, 2.87 with six; 24 of 40 x 36 x 60 (0.2 GB) 120,
    // 106 and 95 us.
    if (op == OP_CONVERT && (long long)total * 256 * 3 * b->meqn * (long long)sizeof(T) > 256ll << 20)
        grid = std::min(grid, 3 * b->ncu);
    HIPCHECK(hipLaunchKernel(fn, dim3(std::min(total, grid)), list_block(lg), kargs, 0, b->stream));
    return launch_check();
}

static GateSpec gs(int mode, int nn = 0, int kk = 0, int fslot = -1) { return GateSpec{mode, nn, kk, fslot}; }

// src3 of the accepted scenarios after its conversion (launch_group):
// src3_passes32 / src3_passes64's sequence
// with the substep loops run to the captured caps, each scenario gated by
// its own counts (src3.f90:203-634, diffuse.f:37-210, conduct.f:245-332)
template <typename T>
static int launch_src(magic_batch *b)
{
    for (int nn = 1; nn <= b->ndtr_cap; nn++) {
        // bc3 with the z faces skipped (src3.f90:333-336) and diffuse's z ghosts
        TRY(launch_op<T>(b, OP_BCUVW, gs(GATE_DIFF, nn)));
        TRY(launch_op<T>(b, OP_DIFF_CROSS, gs(GATE_DIFF, nn, 0, FAC_CROSS)));
        TRY(launch_op<T>(b, OP_DIFF, gs(GATE_DIFF, nn, 1, FAC_DIFF)));
        for (int kk = 2; kk <= b->ndtrc_cap; kk++) TRY(launch_op<T>(b, OP_CONDUCT, gs(GATE_COND, nn, kk, FAC_DIFF), kk));
        if (nn < b->ndtr_cap) TRY(launch_op<T>(b, OP_COPY_T, gs(GATE_MORE, nn)));
    }
    return launch_op<T>(b, OP_FINISH, gs(GATE_ACCEPTED));
}

// The argument blocks of a slot's sweeps moved on to the blocks of a slab
template <typename T>
struct SlabArgs {
    T *parts[3];
    int sT[3], sK[3], sS[3];
};
template <typename T>
__global__ void k_slab_args(SweepArgsT<T> *args, SlabArgs<T> a)
{
    const int d = (int)threadIdx.x;
    if (d >= 3) return;
    args[d].parts = a.parts[d];
    args[d].sT = a.sT[d];
    args[d].sK = a.sK[d];
    args[d].sS = a.sS[d];
}
// Launches it; sp: the slab's increments
template <typename T>
static int put_slab(magic_batch *b, const magic_batch::Group &g, StepParts<T> &sp)
{
    const magic_ctx *c = b->sc[g.lo];
    const Slab &slab = b->slabs[g.lo][g.slab];
    SlabArgs<T> sa;
    T *next = (T *)b->parts;
    sp.nc = c->meqn;
    for (int dir = 0; dir < 3; dir++) {
        SweepArgsT<T> a;
        sweep_geometry(c, dir, b->shape[dir], a, sp.d[dir]);
        next = parts_layout(a, sp.d[dir], dir, slab.lo[dir], slab.hi[dir], c->meqn, b->shape[dir], next);
        sa.parts[dir] = a.parts;
        sa.sT[dir] = a.sT; sa.sK[dir] = a.sK; sa.sS[dir] = a.sS;
    }
    k_slab_args<T><<<1, 64, 0, b->stream>>>((SweepArgsT<T> *)b->args_d + 3 * g.lo, sa);
    return launch_check();
}

// Sweeps, decision and conversion of one group.  A grid in slabs is swept from
// the copied backup and each slab's increments are added to q at once, as one
// grid does (capi.hip).
template <typename T, bool PERT>
static int launch_group(magic_batch *b, const magic_batch::Group &g)
{
    StepParts<T> sp;
    if (g.slab == 0) TRY(launch_op<T>(b, OP_BACKUP, gs(GATE_RUN), 0, g.lo, g.hi));
    if (g.slab >= 0) TRY(put_slab<T>(b, g, sp));
    for (int d0 = 0, d1; d0 < 3; d0 = d1) {
        for (d1 = d0 + 1; d1 < 3 && b->shape[d1] == b->shape[d0];) d1++;
        TRY((launch_dirs<T, PERT>(b, g, d0, d1)));
    }
    if (g.slab >= 0) {
        const magic_ctx *c = b->sc[g.lo];
        const Slab &s = b->slabs[g.lo][g.slab];
        k_add_parts<T><<<slab_cells(c->d, s), cell_block(), 0, b->stream>>>(c->d, state_q(c, T()), sp, s.i0 + c->mbc - 1,
                                                                            s.i1 + c->mbc - 1, &b->ctl_d[g.lo].swept);
        TRY(launch_check());
        if (g.slab + 1 < g.nslab) return MAGIC_OK;
    }
    k_batch_decide<<<blocks(g.hi - g.lo, 256), 256, 0, b->stream>>>(b->ctl_d + g.lo, g.hi - g.lo);
    TRY(launch_check());
    if (g.slab >= 0) TRY(launch_op<T>(b, OP_RESTORE, gs(GATE_DROPPED), 0, g.lo, g.hi));
    return launch_op<T>(b, OP_CONVERT, gs(GATE_ACCEPTED), 0, g.lo, g.hi);
}

// one attempt of every scenario, as launched into the capture
template <typename T, bool PERT>
static int record_attempt(magic_batch *b)
{
    k_batch_prepare<T><<<blocks(b->n, 256), 256, 0, b->stream>>>(b->ctl_d, b->n, (SweepArgsT<T> *)b->args_d);
    TRY(launch_check());
    const GateSpec run = gs(GATE_RUN);
    TRY(launch_op<T>(b, OP_BC, run));   // with b4step3
    TRY(launch_op<T>(b, OP_BCZ, run));            // grids with mz < mbc only
    for (const auto &g : b->groups) TRY((launch_group<T, PERT>(b, g)));
    TRY(launch_src<T>(b));
    k_batch_finalize<<<blocks(b->n, 256), 256, 0, b->stream>>>(b->ctl_d, b->n);
    return launch_check();
}

// Form-specific part of a scenario's sweep argument block
static void sweep_form_args(const magic_ctx *c, SweepArgsT<float> &a)
{
    const int NZ = c->d.NZ;
    a.qold = c->q32;
    a.crho = c->bg64 + B64_RHO * NZ;
    a.cE = c->bg64 + B64_E * NZ;
    a.cgam = c->bg64 + B64_GAM * NZ;
    a.cvg = c->bg64 + B64_VG * NZ;
    a.cres = c->bg64 + B64_RES * NZ;
}

static void sweep_form_args(const magic_ctx *c, SweepArgsT<double> &a)
{
    a.qold = c->q;
    a.gam = c->aux + AX_GAM * c->P;
    a.vgrav = c->aux + AX_VG * c->P;
}

// Room for the increments of a batch's grids.  A batch of more grids than
// this holds runs its sweeps in groups; 8 GB (40 million FP64 cells of six
// components, twice that in FP32) fill the chip many times over, so that the
// groups cost nothing, and the bound keeps the batch's memory near what its
// scenarios' own states take.
constexpr size_t PARTS_BYTES = size_t(8) << 30;

// The part buffer given back; the next list build sets it up again
static void drop_parts(magic_batch *b)
{
    if (!b->parts_of) hipFree(b->parts);
    b->parts = nullptr;
    b->parts_bytes = 0;
    b->parts_of = nullptr;
}

// The part buffer and the groups for the batch's shapes
template <typename T>
static int build_groups(magic_batch *b)
{
    std::vector<size_t> need(b->n, 0);
    size_t sum = 0, big = 0, least = 0;
    magic_ctx *roomy = nullptr;   // the scenario with the largest staging buffer
    for (int s = 0; s < b->n; s++) {
        if (!b->sc[s]) continue;
        if (!roomy || stage_bytes(b->sc[s]) > stage_bytes(roomy)) roomy = b->sc[s];
        const Slabs<T> slabs(b->sc[s], b->shape);
        need[s] = slabs.whole();
        sum += need[s];
        big = std::max(big, need[s]);
        least = std::max(least, slabs.least());
    }
    const size_t want = b->parts_room ? std::min(sum, std::max(least, b->parts_room)) : std::max(big, std::min(sum, PARTS_BYTES));
    if (b->parts_bytes < want) {
        drop_parts(b);
        size_t got = want;
        // less room: smaller groups, then the largest grids in slabs, at last
        // in a staging buffer, idle in an attempt
        while (hipMalloc(&b->parts, got) != hipSuccess) {
            (void)hipGetLastError();
            b->parts = nullptr;
            if (got == least) {
                if (stage_bytes(roomy) < least) return MAGIC_ENOMEM;
                b->parts = roomy->stage;
                b->parts_of = roomy;
                got = stage_bytes(roomy);
                break;
            }
            got = std::max(got > big ? big : least, got / 2);
        }
        b->parts_bytes = got;
    }
    b->groups.clear();
    b->slabs.assign(b->n, {});
    size_t used = 0;
    for (int s = 0; s < b->n; s++) {
        magic_batch::Group g = {s, s + 1, {0, 0, 0, 0}};
        if (need[s] > b->parts_bytes) {
            b->slabs[s] = Slabs<T>(b->sc[s], b->shape).within(b->parts_bytes);
            g.nslab = (int)b->slabs[s].size();
            for (g.slab = 0; g.slab < g.nslab; g.slab++) b->groups.push_back(g);
            continue;
        }
        if (b->groups.empty() || b->groups.back().slab >= 0 || used + need[s] > b->parts_bytes) {
            b->groups.push_back(g);
            used = 0;
        }
        used += need[s];
        b->groups.back().hi = s + 1;
    }
    return MAGIC_OK;
}

// Sweep argument blocks, the groups and their blocks' lists (geometry only;
// the step's dt factors are written by k_batch_prepare).  For the autotuner
// (tuning) every block runs and the dt factors come from each scenario's
// next dt.
template <typename T>
static int build_lists(magic_batch *b, bool tuning = false)
{
    TRY(build_groups<T>(b));
    std::vector<SweepArgsT<T>> args((size_t)b->n * 3);
    std::vector<const int *> run((size_t)b->n * 3);
    std::vector<int4> items;
    b->sp64.assign(b->n, StepParts<double>{});
    b->sp32.assign(b->n, StepParts<float>{});
    for (auto &g : b->groups) {
        T *next = (T *)b->parts;
        for (int dir = 0; dir < 3; dir++) {
            g.off[dir] = (int)items.size();
            for (int s = g.lo; s < g.hi; s++) {
                magic_ctx *c = b->sc[s];
                if (!c) continue;
                SweepArgsT<T> &a = args[3 * s + dir];
                StepParts<T> &sp = slot_parts(b, s, T());
                SweepParts<T> &p = sp.d[dir];
                memset(&a, 0, sizeof(a));
                sweep_form_args(c, a);
                sweep_geometry(c, dir, b->shape[dir], a, p);
                sp.nc = c->meqn;
                a.nspecadv = c->have_params ? c->prm.nspecadv : 0;
                a.cfl_bits = &b->ctl_d[s].cfl_bits;
                a.status = &b->ctl_d[s].err[0];
                if (g.slab >= 0 || tuning) a.qold = (const T *)state_qold(c);
                const double dt = b->ctl[s].dt > 0.0 ? b->ctl[s].dt : 1.0;
                if (tuning) sweep_factors(c, dir, dt, a);
                int lo = 0, hi = dir == 0 ? p.nk : p.nt;
                if (g.slab >= 0) {   // put_slab places its parts
                    lo = b->slabs[s][g.slab].lo[dir];
                    hi = b->slabs[s][g.slab].hi[dir];
                } else {
                    next = parts_layout(a, p, dir, lo, hi, c->meqn, b->shape[dir], next);
                }
                run[3 * s + dir] = tuning ? b->one_d : &b->ctl_d[s].run;
                push_items(items, p, dir, lo, hi, 3 * s + dir);
                if (items.size() > 0x7fffffff) return MAGIC_EUNSUPPORTED;
            }
        }
        g.off[3] = (int)items.size();
    }
    const size_t total = items.size();
    hipFree(b->items_d);
    b->items_d = nullptr;
    if (hipMalloc(&b->items_d, (total ? total : 1) * sizeof(int4)) != hipSuccess) {
        (void)hipGetLastError();
        b->items_d = nullptr;
        return MAGIC_ENOMEM;
    }
    HIPCHECK(hipMemcpyAsync(b->items_d, items.data(), total * sizeof(int4), hipMemcpyHostToDevice, b->stream));
    HIPCHECK(hipMemcpyAsync(b->args_d, args.data(), args.size() * sizeof(args[0]), hipMemcpyHostToDevice, b->stream));
    HIPCHECK(hipMemcpyAsync(b->run_d, run.data(), run.size() * sizeof(run[0]), hipMemcpyHostToDevice, b->stream));
    HIPCHECK(hipStreamSynchronize(b->stream));
    return MAGIC_OK;
}

// Form-specific operands of a scenario's boundary and source-pass kernels
static void form_ops(const magic_ctx *c, BatchOps<float> &o)
{
    const int NZ = c->d.NZ;
    o.q = c->q32; o.qold = c->qold32; o.u = c->u32; o.qt = c->qt32; o.ut = c->ut32;
    o.col = col32_of(c);
    o.zr = c->zr32;
    o.nu32 = c->col32 + C32_NU * NZ;
    o.kap32 = c->col32 + C32_KAP * NZ;
}

static void form_ops(const magic_ctx *c, BatchOps<double> &o)
{
    const int NZ = c->d.NZ;
    const long long P = c->P;
    o.q = c->q; o.qold = c->qold; o.u = c->u; o.qt = c->qt; o.ut = c->ut;
    const double *A = c->col64;   // the background's columns (magic_batch_start checks they exist)
    o.ax = {A + AX_RHO * NZ, A + AX_MX * NZ, A + AX_MY * NZ, A + AX_MZ * NZ, A + AX_E * NZ, A + AX_R * NZ,
            A + AX_GAM * NZ};
    o.nu64 = A + AX_NU * NZ;
    o.kap64 = A + AX_KAP * NZ;
    o.aux1 = c->aux + AX_RHO * P;
    o.aux2 = c->aux + AX_MX * P;
    o.aux3 = c->aux + AX_MY * P;
    o.aux5 = c->aux + AX_E * P;
    o.zratio = c->zratio;
}

// Layers per workgroup of the diffusion kernels of a batch.  A workgroup forms
// the two layers around its own as well; one grid takes few layers (diff_kb)
// to have enough workgroups, a batch has them from its scenarios: about 4096, of
// 8 to 16 layers (24 FP32 grids of 40 x 36 x 60: the passes 68 us with 16
// layers, 49 with 4, 45 with 8).  The result does not depend on the layer count.
static int batch_kb(const magic_batch *b)
{
    long long work = 0;
    for (const magic_ctx *c : b->sc)
        if (c) work += 4ll * passes_cols(c->d).x * passes_cols(c->d).y * c->mz;
    return (int)std::min<long long>(16, std::max<long long>(8, work / 4096));
}

// whether a scenario's z faces run after the others in their own pass (capi.hip's bc_launch)
static bool z_apart(const magic_ctx *c, const int *bc) { return c->mz < c->mbc && (bc[4] > 0 || bc[5] > 0); }

// Grid of list lg for one scenario (x, y, z blocks; x = 0: no blocks)
static int4 list_grid(const magic_batch *b, const magic_ctx *c, const int *bc, int lg, int kb)
{
    const Dims &d = c->d;
    const long long P = c->P;
    auto g1 = [](long long x) { return make_int4((int)x, 1, 1, 0); };
    const int nzb = (int)blocks(d.mz, kb);
    switch (lg) {
    case LG_BC: case LG_BCUVW: {
        long long n = (long long)bc_lanes(d, 0) + bc_lanes(d, 1) + bc_lanes(d, 2);
        if (lg == LG_BC && b->meqn > 5) n += bc_lanes(d, 3);
        return g1(blocks(n, 256));
    }
    case LG_BCZ: return z_apart(c, bc) ? make_int4(blocks(d.NX, 64), d.NY, 1, 0) : g1(0);
    case LG_CPY: return g1(std::min<long long>(8192, blocks(P * b->meqn, 256)));
    case LG_PAD: { const dim3 g = padded_cells(d); return make_int4(g.x, g.y, g.z, 0); }
    case LG_DIF: return make_int4(diff_cols(d).x, diff_cols(d).y, nzb, 0);
    case LG_DF1: case LG_DF4: return make_int4(passes_cols(d).x, passes_cols(d).y, (lg == LG_DF4 ? 4 : 1) * nzb, 0);
    case LG_INT: { const dim3 g = interior_grid(d); return make_int4(g.x, g.y, g.z, 0); }
    default: return g1(0);
    }
}

// Operand blocks and block lists of the boundary, copy and source-pass
// kernels, and the substep loops the capture records
template <typename T>
static int build_ops(magic_batch *b)
{
    const int kb = batch_kb(b);
    std::vector<BatchOps<T>> ops(b->n);
    std::vector<int> off((size_t)NLG * (b->cap + 1), 0);
    std::vector<int4> gdim((size_t)NLG * b->cap, make_int4(0, 1, 1, 0));
    b->ndtr_cap = 0;
    b->ndtrc_cap = 0;
    for (int lg = 0; lg < NLG; lg++) {
        long long total = 0;
        for (int s = 0; s < b->n; s++) {
            off[(size_t)lg * (b->cap + 1) + s] = (int)total;
            magic_ctx *c = b->sc[s];
            if (!c) continue;
            const int4 g = list_grid(b, c, &b->mthbc[6 * s], lg, kb);
            gdim[(size_t)lg * b->cap + s] = g;
            total += (long long)g.x * g.y * g.z;
            if (total > 0x7fffffff) return MAGIC_EUNSUPPORTED;
        }
        off[(size_t)lg * (b->cap + 1) + b->n] = (int)total;
    }
    for (int s = 0; s < b->n; s++) {
        magic_ctx *c = b->sc[s];
        BatchOps<T> &o = ops[s];
        memset(&o, 0, sizeof(o));
        o.ctl = b->ctl_d + s;   // an empty slot's control block is all zeros: every gate off
        if (!c) continue;
        o.d = c->d;
        form_ops(c, o);
        o.sp = slot_parts(b, s, T());
        o.added = !b->slabs[s].empty();
        o.nc = c->meqn;
        o.kb = kb;
        o.spill = c->mz > c->mx ? c->mz - c->mx : 0;
        for (int f = 0; f < 6; f++) o.bc.m[f] = std::max(0, b->mthbc[6 * s + f]);
        o.bcz = z_apart(c, &b->mthbc[6 * s]);
        const magic_params &p = c->prm;
        Forcing &f = o.f;
        f.forcemth = (int)p.forcemth;
        f.t = 0.0; f.dt = 0.0; f.tgauss = 0.0;   // from the control block at run time
        f.xlower = c->xlower; f.ylower = c->ylower; f.zlower = c->zlower;
        f.dx = c->dx; f.dy = c->dy; f.dz = c->dz;
        f.amplitude = p.amplitude; f.xpos = p.xpos; f.ypos = p.ypos; f.zpos = p.zpos;
        f.xwidth = p.xwidth; f.ywidth = p.ywidth; f.zwidth = p.zwidth;
        f.tcenter = p.tcenter; f.twidth = p.twidth;
        f.omega = p.omega; f.propx = p.propx; f.propz = p.propz; f.vsrcx = p.vsrcx;
        b->ndtr_cap = std::max(b->ndtr_cap, b->ctl[s].ndtr_cap);
        b->ndtrc_cap = std::max(b->ndtrc_cap, b->ctl[s].ndtrc_cap);
    }
    b->loff = off;
    HIPCHECK(hipMemcpyAsync(b->ops_d, ops.data(), ops.size() * sizeof(ops[0]), hipMemcpyHostToDevice, b->stream));
    HIPCHECK(hipMemcpyAsync(b->loff_d, off.data(), off.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
    HIPCHECK(hipMemcpyAsync(b->lgdim_d, gdim.data(), gdim.size() * sizeof(int4), hipMemcpyHostToDevice, b->stream));
    HIPCHECK(hipStreamSynchronize(b->stream));
    return MAGIC_OK;
}

// persistent grid of each kernel class of the work-list launches: as many
// workgroups as fit on the chip at once
template <typename T>
static int list_grids(magic_batch *b)
{
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    HIPCHECK(hipDeviceGetAttribute(&b->ncu, hipDeviceAttributeMultiprocessorCount, dev));
    for (int op = 0; op < NOP; op++) {
        const void *fn = batch_op_fn<T>(op);
        if (!fn) return MAGIC_EUNSUPPORTED;
        const dim3 blk = list_block(op_list(op));
        int occ = 0;
        HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, (int)(blk.x * blk.y * blk.z), 0));
        b->opgrid[op] = b->ncu * (occ > 0 ? occ : 1);
    }
    return MAGIC_OK;
}

// Retire the captured attempt: wait until no replay runs, then destroy the executable graph and
// the graph itself.  Called before any device buffer its kernels address
// (control blocks, argument blocks, work and block lists, a scenario's
// state) is freed or reallocated, so that no instantiated graph ever holds
// a dangling pointer, and before every capture.
static int drop_graph(magic_batch *b)
{
    int st = MAGIC_OK;
    if (b->stream && hipStreamSynchronize(b->stream) != hipSuccess) st = MAGIC_EHIP;
    if (b->exec) hipGraphExecDestroy(b->exec);
    if (b->graph) hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->graph_ok = false;
    return st;
}

template <typename T, bool PERT>
static int build_graph_t(magic_batch *b)
{
    TRY(drop_graph(b));
    TRY(list_grids<T>(b));
    TRY(build_lists<T>(b));
    TRY(build_ops<T>(b));
    HIPCHECK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    const int st = record_attempt<T, PERT>(b);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(b->stream, &g);
    if (st != MAGIC_OK) {
        if (g) hipGraphDestroy(g);
        return st;
    }
    HIPCHECK(e);
    b->graph = g;
    HIPCHECK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    b->graph_ok = true;
    return MAGIC_OK;
}

static int build_graph(magic_batch *b)
{
    return fp32(b) ? build_graph_t<float, true>(b) : build_graph_t<double, false>(b);
}

// ------------------------------------------------------------------ ABI --
// device arrays for at least want slots (contents are rebuilt from the host
// copies before the next attempt)
static int reserve(magic_batch *b, int want)
{
    if (want <= b->cap) return MAGIC_OK;
    int cap = b->cap ? b->cap : 8;
    while (cap < want) cap *= 2;
    TRY(drop_graph(b));
    hipFree(b->ctl_d); hipFree(b->args_d); hipFree(b->run_d);
    hipFree(b->ops_d); hipFree(b->loff_d); hipFree(b->lgdim_d);
    if (b->ctl_pin) hipHostFree(b->ctl_pin);
    b->ctl_d = nullptr; b->args_d = nullptr; b->run_d = nullptr; b->ctl_pin = nullptr;
    b->ops_d = nullptr; b->loff_d = nullptr; b->lgdim_d = nullptr;
    b->cap = 0;
    const size_t args_bytes = fp32(b) ? sizeof(SweepArgsT<float>) : sizeof(SweepArgsT<double>);
    const size_t ops_bytes = fp32(b) ? sizeof(BatchOps<float>) : sizeof(BatchOps<double>);
    if (hipMalloc(&b->ctl_d, cap * sizeof(ScenCtl)) != hipSuccess ||
        hipHostMalloc(&b->ctl_pin, cap * sizeof(ScenCtl), hipHostMallocDefault) != hipSuccess ||
        hipMalloc(&b->args_d, (size_t)cap * 3 * args_bytes) != hipSuccess ||
        hipMalloc(&b->run_d, (size_t)cap * 3 * sizeof(int *)) != hipSuccess ||
        hipMalloc(&b->ops_d, (size_t)cap * ops_bytes) != hipSuccess ||
        hipMalloc(&b->loff_d, (size_t)NLG * (cap + 1) * sizeof(int)) != hipSuccess ||
        hipMalloc(&b->lgdim_d, (size_t)NLG * cap * sizeof(int4)) != hipSuccess)
        return MAGIC_ENOMEM;
    b->cap = cap;
    b->graph_ok = false;
    b->dirty = true;
    return MAGIC_OK;
}

extern "C" int magic_batch_add(magic_batch *b, const int dims[3], const double geom[6], int *slot)
{
    if (!b || !dims || !geom || !slot) return MAGIC_EARG;
    magic_ctx *c = nullptr;
    TRY(magic_create_form(dims[0], dims[1], dims[2], b->meqn, b->mbc, b->maux, geom[0], geom[1], geom[2],
                          geom[3], geom[4], geom[5], b->form, &c));
    hipStreamSynchronize(c->stream);
    hipStreamDestroy(c->stream);
    c->stream = b->stream;
    c->own_stream = false;
    int s = 0;
    while (s < b->n && b->sc[s]) s++;
    if (s == BATCH_MAX_SLOTS) {
        magic_destroy(c);
        return MAGIC_EUNSUPPORTED;
    }
    if (s == b->n) {
        const int st = reserve(b, b->n + 1);
        if (st != MAGIC_OK) {
            magic_destroy(c);
            return st;
        }
        b->n++;
        b->sc.push_back(nullptr);
        b->ctl.push_back(ScenCtl());
        b->mthbc.insert(b->mthbc.end(), 6, 1);
        b->settled.push_back(0);
    }
    b->sc[s] = c;
    memset(&b->ctl[s], 0, sizeof(ScenCtl));   // inactive until started
    b->graph_ok = false;
    b->dirty = true;
    *slot = s;
    return MAGIC_OK;
}

extern "C" int magic_batch_remove(magic_batch *b, int s)
{
    if (!b || s < 0 || s >= b->n || !b->sc[s]) return MAGIC_EARG;
    TRY(drop_graph(b));
    if (b->parts_of == b->sc[s]) drop_parts(b);
    magic_destroy(b->sc[s]);
    b->sc[s] = nullptr;
    memset(&b->ctl[s], 0, sizeof(ScenCtl));
    b->graph_ok = false;
    b->dirty = true;
    return MAGIC_OK;
}

extern "C" int magic_batch_create(int nscen, const int *dims, int meqn, int mbc, int maux, const double *geom,
                                  int form, magic_batch **out)
{
    if (!out || nscen < 0 || (nscen > 0 && (!dims || !geom))) return MAGIC_EARG;
    *out = nullptr;
    if (form != MAGIC_FORM_FP32P && form != MAGIC_FORM_FP64) return MAGIC_EUNSUPPORTED;
    if (mbc < 2 || mbc > 8 || meqn < 5 || meqn > 10 || maux < 19) return MAGIC_EARG;
    if (!sweep_supported(meqn - 5)) return MAGIC_EUNSUPPORTED;
    magic_batch *b = new magic_batch();
    b->meqn = meqn;
    b->mbc = mbc;
    b->maux = maux;
    b->form = form;
    int st = MAGIC_OK;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) st = MAGIC_EHIP;
    if (st == MAGIC_OK) st = reserve(b, nscen > 0 ? nscen : 1);
    if (st == MAGIC_OK) st = hipMalloc(&b->one_d, sizeof(int)) == hipSuccess ? MAGIC_OK : MAGIC_ENOMEM;
    if (st == MAGIC_OK) {
        const int one = 1;
        st = hipMemcpy(b->one_d, &one, sizeof(int), hipMemcpyHostToDevice) == hipSuccess ? MAGIC_OK : MAGIC_EHIP;
    }
    for (int s = 0; s < nscen && st == MAGIC_OK; s++) {
        int slot;
        st = magic_batch_add(b, dims + 3 * s, geom + 6 * s, &slot);
    }
    if (st != MAGIC_OK) {
        magic_batch_destroy(b);
        return st;
    }
    *out = b;
    return MAGIC_OK;
}

extern "C" int magic_batch_destroy(magic_batch *b)
{
    if (!b) return MAGIC_OK;
    drop_graph(b);
    drop_parts(b);
    for (auto c : b->sc)
        if (c) magic_destroy(c);
    hipFree(b->ctl_d); hipFree(b->args_d); hipFree(b->run_d); hipFree(b->items_d);
    hipFree(b->one_d); hipFree(b->ops_d); hipFree(b->loff_d); hipFree(b->lgdim_d);
    if (b->ctl_pin) hipHostFree(b->ctl_pin);
    if (b->stream) hipStreamDestroy(b->stream);
    delete b;
    return MAGIC_OK;
}

extern "C" int magic_batch_ctx(magic_batch *b, int s, magic_ctx **ctx)
{
    if (!b || !ctx || s < 0 || s >= b->n || !b->sc[s]) return MAGIC_EARG;
    *ctx = b->sc[s];
    b->graph_ok = false;   // the caller may change parameters, aux or q
    return MAGIC_OK;
}

extern "C" int magic_batch_start(magic_batch *b, int s, double t, double tend, double dt, const double dtv[5],
                                 const double cflv[4], int maxsteps, const int mthbc[6])
{
    if (!b || s < 0 || s >= b->n || !b->sc[s] || !dtv || !cflv || !mthbc || maxsteps < 1) return MAGIC_EARG;
    magic_ctx *c = b->sc[s];
    if (!c->have_aux || !c->have_params) return MAGIC_EARG;
    if (cflv[1] > cflv[0]) return MAGIC_EARG;
    for (int f = 0; f < 6; f++)
        if (mthbc[f] == 0 || mthbc[f] >= 4) return MAGIC_EBC;
    const magic_params &p = c->prm;
    if (p.omega1 != 0.0 || !(p.forcemth == 0.0 || p.forcemth == 1.0 || p.forcemth == 3.0))
        return MAGIC_EUNSUPPORTED;
    // the FP64 form's batched source pass reads the background as columns
    if (!fp32(b) && !c->aux_layered) return MAGIC_EUNSUPPORTED;
    ScenCtl &h = b->ctl[s];
    if (memcmp(&b->mthbc[6 * s], mthbc, 6 * sizeof(int)) != 0) b->graph_ok = false;
    memcpy(&b->mthbc[6 * s], mthbc, 6 * sizeof(int));
    h.t = t;
    h.told = t;
    h.tend = tend;
    h.clip = t < tend;
    h.dt = dt;
    h.dtmax = dtv[1];
    h.cflv1 = cflv[0];
    h.cflv2 = cflv[1];
    h.cfl = 0.0;
    h.cflmax = 0.0;
    h.active = 1;
    h.newstep = 1;
    h.nsteps = 0;
    h.attempts = 0;
    h.rejects = 0;
    h.maxsteps = maxsteps;
    h.status = 0;
    b->settled[s] = 0;
    h.dx = c->dx; h.dy = c->dy; h.dz = c->dz;
    double dmin = c->dx < c->dy ? c->dx : c->dy;
    dmin = dmin < c->dz ? dmin : c->dz;
    h.dxyzmin2 = dmin * dmin;
    h.difmax = (4.0 / 3.0) * c->aux11_top;
    h.kapmax = c->aux12_top;
    h.tcenter = p.tcenter;
    h.twidth = p.twidth;
    int a, bb;
    src_caps(c, dt > dtv[1] ? dt : dtv[1], &a, &bb);
    // the captured substep loops cover every count up to the batch's largest
    if (a > b->ndtr_cap || bb > b->ndtrc_cap) b->graph_ok = false;
    h.ndtr_cap = a;
    h.ndtrc_cap = bb;
    b->dirty = true;
    return MAGIC_OK;
}

extern "C" int magic_batch_run(magic_batch *b, int max_attempts, int check_every, int *attempts_done)
{
    if (!b || max_attempts < 1 || check_every < 1) return MAGIC_EARG;
    if (attempts_done) *attempts_done = 0;
    bool started = false;
    for (int s = 0; s < b->n; s++) started = started || (b->sc[s] && b->ctl[s].active && b->ctl[s].status == 0);
    if (!started) return MAGIC_OK;
    if (!b->graph_ok) {
        // the captured kernels read the control blocks; upload before building
        HIPCHECK(hipMemcpyAsync(b->ctl_d, b->ctl.data(), b->n * sizeof(ScenCtl), hipMemcpyHostToDevice, b->stream));
        TRY(build_graph(b));
        b->dirty = false;
    }
    if (b->dirty) {
        HIPCHECK(hipMemcpyAsync(b->ctl_d, b->ctl.data(), b->n * sizeof(ScenCtl), hipMemcpyHostToDevice, b->stream));
        b->dirty = false;
    }
    if (b->parts_of) TRY(stage_ready(b->parts_of));   // a snapshot may still be copied out of it
    int done = 0;
    bool any = true;
    while (done < max_attempts && any) {
        const int k = std::min(check_every, max_attempts - done);
        for (int i = 0; i < k; i++) HIPCHECK(hipGraphLaunch(b->exec, b->stream));
        done += k;
        HIPCHECK(hipMemcpyAsync(b->ctl_pin, b->ctl_d, b->n * sizeof(ScenCtl), hipMemcpyDeviceToHost, b->stream));
        HIPCHECK(hipStreamSynchronize(b->stream));
        memcpy(b->ctl.data(), b->ctl_pin, b->n * sizeof(ScenCtl));
        any = false;
        for (int s = 0; s < b->n; s++) any = any || (b->ctl[s].active && b->ctl[s].status == 0);
    }
    if (attempts_done) *attempts_done = done;
    // a scenario that failed (rho <= 0, a**2 <= 0, more substeps than
    // captured) has stopped with its status in its control block, which
    // magic_batch_state reports; the others went on
    for (int s = 0; s < b->n; s++)
        if (b->sc[s] && !b->settled[s] && (b->ctl[s].status == MAGIC_ERHO || b->ctl[s].status == MAGIC_EA2)) {
            b->settled[s] = 1;
            TRY(failed_step(b->sc[s], b->shape, b->ctl[s].dt));
        }
    return MAGIC_OK;
}

extern "C" int magic_batch_state(magic_batch *b, int s, double real_out[5], int int_out[6])
{
    if (!b || s < 0 || s >= b->n || !b->sc[s]) return MAGIC_EARG;
    const ScenCtl &h = b->ctl[s];
    if (real_out) {
        real_out[0] = h.t;
        real_out[1] = h.dt;
        real_out[2] = h.cfl;
        real_out[3] = h.cflmax;
        real_out[4] = h.tend;
    }
    if (int_out) {
        int_out[0] = h.nsteps;
        int_out[1] = h.attempts;
        int_out[2] = h.rejects;
        int_out[3] = h.active;
        int_out[4] = h.status;
        int_out[5] = h.ndtr;
    }
    return MAGIC_OK;
}

extern "C" int magic_batch_set_tile_shapes(magic_batch *b, const int shapes[3])
{
    if (!b || !shapes || !shapes_valid(shapes)) return MAGIC_EARG;
    for (int k = 0; k < 3; k++) b->shape[k] = shapes[k];
    b->graph_ok = false;
    return MAGIC_OK;
}

extern "C" int magic_batch_set_increment_room(magic_batch *b, size_t bytes)
{
    if (!b) return MAGIC_EARG;
    TRY(drop_graph(b));   // its kernels hold the buffer's address
    b->parts_room = bytes;
    drop_parts(b);
    return MAGIC_OK;
}

extern "C" int magic_batch_set_sweep_overlap(magic_batch *b, int) { return b ? MAGIC_OK : MAGIC_EARG; }

extern "C" int magic_batch_get_tile_shapes(magic_batch *b, int shapes[3])
{
    if (!b || !shapes) return MAGIC_EARG;
    for (int k = 0; k < 3; k++) shapes[k] = b->shape[k];
    return MAGIC_OK;
}

// Every candidate reads q and writes its own increment blocks (one list
// build per shape and round, all directions), so the states do not change.
// The candidates' Courant numbers and reports land in the control blocks'
// reduction fields, which the next attempt's prepare clears.
template <typename T, bool PERT>
static int tune_rounds(magic_batch *b, int reps, TuneClock &clk)
{
    for (int r = 0; r <= reps; r++) {   // repetition 0 warms up and is not timed
        for (int sh = 0; sh < TILE_NSHAPE; sh++) {
            for (int k = 0; k < 3; k++) b->shape[k] = sh;
            TRY(build_lists<T>(b, true));
            if (b->parts_of) TRY(stage_ready(b->parts_of));
            for (int dir = 0; dir < 3; dir++) {
                TRY(clk.mark(dir, sh, 0, b->stream));
                for (const auto &g : b->groups) {
                    StepParts<T> sp;
                    if (g.slab >= 0) TRY(put_slab<T>(b, g, sp));
                    TRY((launch_dirs<T, PERT>(b, g, dir, dir + 1)));
                }
                TRY(clk.mark(dir, sh, 1, b->stream));
            }
        }
        if (r > 0) TRY(clk.add_round());
    }
    return MAGIC_OK;
}

extern "C" int magic_batch_tune(magic_batch *b, int reps, int shapes_out[3], float *ms_out)
{
    if (!b || reps < 1) return MAGIC_EARG;
    bool any = false;
    for (int s = 0; s < b->n; s++) any = any || b->sc[s] != nullptr;
    if (!any) return MAGIC_EARG;
    TuneClock clk;
    if (!clk.ok) return MAGIC_EHIP;
    const int saved[3] = {b->shape[0], b->shape[1], b->shape[2]};
    TRY(drop_graph(b));   // the lists and argument blocks are rebuilt before the next attempt
    int st = MAGIC_OK;
    for (int s = 0; s < b->n && st == MAGIC_OK; s++)
        if (b->sc[s]) st = tune_state(b->sc[s]);
    if (st == MAGIC_OK) st = fp32(b) ? tune_rounds<float, true>(b, reps, clk) : tune_rounds<double, false>(b, reps, clk);
    for (int s = 0; s < b->n; s++) {
        const int sd = b->sc[s] ? tune_done(b->sc[s]) : MAGIC_OK;
        if (st == MAGIC_OK) st = sd;
    }
    if (st == MAGIC_OK && hipStreamSynchronize(b->stream) != hipSuccess) st = MAGIC_EHIP;
    if (st != MAGIC_OK) {
        for (int k = 0; k < 3; k++) b->shape[k] = saved[k];
        return st;
    }
    int best[3];
    clk.result(reps, best, ms_out);
    for (int k = 0; k < 3; k++) {
        b->shape[k] = best[k];
        if (shapes_out) shapes_out[k] = best[k];
    }
    return MAGIC_OK;
}
