// Boundary, pre-step, copy and source-pass kernels of the batched driver as
// work-list launches: one launch of a kernel class covers every scenario of
// a batch.  The list's blocks are the scenarios' own grids laid end to end
// (scenario s owns blocks off[s] .. off[s+1]-1, a grid of gdim[s] blocks); a
// persistent grid walks the list, finds each block's scenario by a binary
// search over off and runs the single-grid kernel's body (stencil_body.h,
// bc_src.hip, bc_src32.hip) on that scenario's operands, gated by its
// step-control block (batch.h).  The number of launches per attempt does not
// depend on the number of scenarios, and a scenario whose gate is off (not
// running, or past its own substep counts) costs next to nothing.
//
// The kernel template is defined here and instantiated in bc_src32.hip (FP32
// form) and bc_src.hip (FP64 form), each under its form's floating-point
// contraction setting, so a scenario rounds exactly as the same grid stepped
// alone.
#pragma once
#include "batch.h"
#include "bc_src.h"
#include "parts.h"
#include "stencil_body.h"

namespace magic {

// The operands of one scenario (device array, one entry per batch slot).
template <typename T>
struct BatchOps {
    Dims d;
    T *q, *qold, *u, *qt, *ut;
    StepParts<T> sp;  // the sweeps' increments, added in the conversion
    int added;        // they are in q already: the grid is swept in slabs
    int nc;          // meqn
    int kb;          // layers per block of the diffusion kernels (diff_kb)
    int spill;       // conduct.f:86-91 out-of-row writes (mz - mx when mz > mx, else 0)
    Faces bc;        // bc3's faces (the source pass's substeps skip z)
    int bcz;         // the z faces run apart, after the others (mz < mbc)
    ScenCtl *ctl;
    // FP32 form: background columns, z-face factors, diffusivity columns
    Col32 col;
    Zr32 zr;
    const float *nu32, *kap32;
    // FP64 form: background columns (source pass), aux planes and z factors (bc3)
    Aux ax;
    const double *nu64, *kap64, *aux1, *aux2, *aux3, *aux5, *zratio;
    Forcing f;       // t, dt and the time factor come from the control block
};

// Kernel classes of the batched attempt
enum {
    OP_BC = 0, OP_BCUVW, OP_BCZ, OP_BACKUP, OP_RESTORE, OP_CONVERT, OP_DIFF_CROSS, OP_DIFF, OP_CONDUCT, OP_COPY_T, OP_FINISH,
    NOP
};
// Block lists, one per launch geometry:
//   BC  boundary lanes and, with tracers, the interior's (1-D, 256 lanes)
//   BCUVW boundary lanes (1-D, 256 lanes)
//   BCZ bc3 z faces of grids with mz < mbc   (NX/64, NY)
//   CPY grid-stride copy of meqn planes       PAD padded cells     (NX/64, NY/4, NZ)
//   DIF cross terms      (mx/64, my/4, mz/kb)
//   DF1 conduct's substeps kk >= 2  (mx/64, my/(4 DIFF_ROWS), mz/kb)
//   DF4 directional passes of four components, conduct's first substep among them
//       (mx/64, my/(4 DIFF_ROWS), 4 * mz/kb)
//   INT interior cells   (mx/64, my/4, mz)
enum { LG_BC = 0, LG_BCUVW, LG_BCZ, LG_CPY, LG_PAD, LG_DIF, LG_DF1, LG_DF4, LG_INT, NLG };

struct GateSpec {
    int mode, nn, kk, fslot;
};

// Slots a batch may hold (the work-list kernels keep one offset per slot in
// LDS)
constexpr int BATCH_MAX_SLOTS = 2048;

// The slot of active block a: the largest s with pre[s] <= a (slots with
// no active blocks, whose pre equals the next slot's, are passed over)
__device__ __forceinline__ int active_find(const int *pre, int n, int a)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= a) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// T' after the substeps: conduct's last one wrote ut (odd count) or qt; with no
// substep it is still q's own plane
template <typename T>
__device__ __forceinline__ const T *conducted(const BatchOps<T> &o, const StepGate &g)
{
    const int n = g.c->ndtr > 0 ? g.c->ndtrc : 0;
    return n == 0 ? o.q + 4 * o.d.P : (n & 1) ? o.ut : o.qt;
}

// One launch of kernel class OP over the blocks of the scenarios' list
// (off, gdim) whose gates are on.  Each workgroup of the persistent grid
// first evaluates every slot's gate and lays the active slots' blocks end to
// end in LDS (pre: active blocks before each slot), then takes active
// blocks blockIdx.x, blockIdx.x + gridDim.x, ...; a launch whose gates are
// all off ends after that scan.  arg: conduct's substep of
// OP_CONDUCT.  The form's own bodies
// are reached through the FORM functor (FP32: bc_src32.hip, FP64:
// bc_src.hip).  n <= BATCH_MAX_SLOTS (the host checks).
template <typename T, int OP, class FORM>
__global__ __launch_bounds__(256) void k_batch_op(const BatchOps<T> *__restrict__ S, const int *__restrict__ off,
                                                  const int4 *__restrict__ gdim, int n, GateSpec gs, int arg)
{
    // No kernel of an attempt writes the operand blocks or the lists, and
    // only prepare, decide and finalize write the control blocks: read
    // through the constant address space, their values stay in scalar
    // registers although the bodies store to q between the reads.
    const cptr<BatchOps<T>> CS = (cptr<BatchOps<T>>)S;
    const cptr<int> coff = (cptr<int>)off;
    const cptr<int> cgdim = (cptr<int>)gdim;   // 4 ints per scenario
    __shared__ int pre[BATCH_MAX_SLOTS + 1];
    __shared__ int wsum[4];
    {
        // thread t owns slots t*per .. t*per+per-1: their active block
        // counts go to pre, then their exclusive prefix replaces them
        const int t = (int)(threadIdx.y * blockDim.x + threadIdx.x);
        const int nt = (int)(blockDim.x * blockDim.y);   // 64 or 256 lanes
        const int per = (n + nt - 1) / nt;
        int sum = 0;
        for (int i = 0; i < per; i++) {
            const int sl = t * per + i;
            if (sl >= n) break;
            // a slot with no blocks here (an empty slot among them) is not
            // looked at further
            int c = coff[sl + 1] - coff[sl];
            if (c > 0) {
                const StepGate g = {(cptr<ScenCtl>)CS[sl].ctl, gs.mode, gs.nn, gs.kk, gs.fslot};
                if (!g.on()) c = 0;
            }
            pre[sl] = c;
            sum += c;
        }
        const int lane = t & 63, wave = t >> 6;
        int v = sum;   // inclusive scan over the wave
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(v, d, 64);
            if (lane >= d) v += y;
        }
        if (lane == 63) wsum[wave] = v;
        __syncthreads();
        int acc = v - sum;
        for (int w = 0; w < wave; w++) acc += wsum[w];
        for (int i = 0; i < per; i++) {
            const int sl = t * per + i;
            if (sl >= n) break;
            const int c = pre[sl];
            pre[sl] = acc;
            acc += c;
        }
        if (t == nt - 1) pre[n] = acc;
        __syncthreads();
    }
    const int total = pre[n];
    const int G = (int)gridDim.x;
    int s = 0, lo = 0, hi = 0;   // the current slot and its active blocks [lo, hi)
    for (int b = (int)blockIdx.x; b < total; b += G) {
        if (b < lo || b >= hi) {
            s = __builtin_amdgcn_readfirstlane(active_find(pre, n, b));
            lo = __builtin_amdgcn_readfirstlane(pre[s]);
            hi = __builtin_amdgcn_readfirstlane(pre[s + 1]);
        }
        const BatchOps<T> o = cload(CS + s);
        const StepGate g = {(cptr<ScenCtl>)o.ctl, gs.mode, gs.nn, gs.kk, gs.fslot};
        const int l = b - lo;
        const int gx = cgdim[4 * s], gy = cgdim[4 * s + 1];
        const uint3 bi = make_uint3((unsigned)(l % gx), (unsigned)((l / gx) % gy), (unsigned)(l / (gx * gy)));
        const long long P = o.d.P;
        if constexpr (OP == OP_BC || OP == OP_BCUVW) {
            // the boundary pass of a step, or of a diffusion substep, which skips z
            Faces f = o.bc;
            if (OP == OP_BCUVW || o.bcz) f.m[4] = f.m[5] = 0;
            b_bc(bi, o.d, o.q, o.nc, f, OP == OP_BC ? CLAMP_BC : UVW_BC, FORM::zscale(o, CS + s), g);
        } else if constexpr (OP == OP_BCZ) {
            FORM::bc_z(bi, o, CS + s, g);
        } else if constexpr (OP == OP_BACKUP) {
            b_copy(bi, (unsigned)gx, o.qold, o.q, P * o.nc, g);
        } else if constexpr (OP == OP_RESTORE) {
            b_copy(bi, (unsigned)gx, o.q, o.qold, P * o.nc, g);
        } else if constexpr (OP == OP_CONVERT) {
            FORM::convert(bi, o, g);
        } else if constexpr (OP == OP_DIFF_CROSS) {
            b_diff_cross<T, true>(bi, o.d, o.u, o.q, FORM::nu(o), T(0.0), T(0.0), T(0.0), o.kb, g);
            __syncthreads();   // the next block's writers of the tile arrays wait for this one's readers
        } else if constexpr (OP == OP_DIFF || OP == OP_CONDUCT) {
            // arg (OP_CONDUCT): the substep kk >= 2
            const DiffArgs<T> a = {o.q, o.u, o.ut, o.qt, FORM::nu(o), FORM::kap(o), {}, o.spill, o.kb};
            b_diff<T, true>(bi, o.d, a, [&](int i) { return g.f(T(0.0), i); }, OP == OP_DIFF ? 1 : arg, g);
        } else if constexpr (OP == OP_COPY_T) {
            b_copy_interior(bi, o.d, o.q + 4 * P, conducted(o, g), 1, g);
        } else if constexpr (OP == OP_FINISH) {
            FORM::finish(bi, o, g);
        }
    }
}

// The kernel of class op for form T (FP32: float, FP64: double), defined by
// the form's source file.
template <typename T>
const void *batch_op_fn(int op);

}  // namespace magic
