// Boundary and source-pass kernels of the FP32 perturbation form.
//
// The state is q' = q - q_bar on component planes (float), with a
// background column at rest: q_bar = (rho_bar(k), 0, 0, 0, E_bar(k)) and
// p_bar = (gamma-1) E_bar.  Tracers are stored as they are (their background
// is 0).  Every formula below is the FP64 form's operator (bc_src.hip, the
// reference's bc3_mpi.f / src3.f90) rewritten so that no FP32 operation
// subtracts two background-sized numbers.  Products and sums may contract
// into fused multiply-adds: this form's error bar is a fraction of the field
// peak against the FP64 form.
#pragma clang fp contract(fast)
#include "batch.h"
#include "magic_dev.h"
#include "stencil_body.h"
#include "batch_ops.h"

namespace magic {

// FP32 instantiations of the shared kernels (coefficients as columns)
template __global__ void k_bc<float, ZScale32, GridGate>(Dims, float *, int, Faces, int, ZScale32, GridGate);
template __global__ void k_diff<float, true, GridGate>(Dims, DiffArgs<float>, int, GridGate);
template __global__ void k_clamp<float, GridGate>(float *, long long, int, GridGate);
template __global__ void k_diff_cross<float, true, GridGate>(Dims, float *, const float *, const float *, float, float, float,
                                                        int, GridGate);
template __global__ void k_copy_interior<float, GridGate>(Dims, float *, const float *, int, GridGate);
// z faces (bc3_mpi.f:544-809).  The FP64 form writes
//   q_ghost = aux_ghost + (q_boundary - aux_boundary) * sc
// for rho, the horizontal momenta and E, and q_ghost = q_boundary * sc for
// the vertical momentum; with a background at rest every one of them is
// q'_ghost = q'_boundary * sc.  sc depends on the layer only.
// zf(side, kbc - 1): the factor sc of ghost layer kbc on side 0 (bottom) or 1
// (top), Zr32's s[side][kbc - 1] (FP64)
template <class G, class ZF>
__device__ __forceinline__ void b32_bc_z(const uint3 BI, Dims d, float *q, int nc, int lo, int hi, ZF zf,
                                         const G &gate)
{
    if (!gate.on()) return;
    const int i = (int)(BI.x * blockDim.x + threadIdx.x) + 1 - d.mbc;
    const int j = (int)BI.y + 1 - d.mbc;
    if (i > d.mx + d.mbc || j > d.my + d.mbc) return;
    for (int side = 0; side < 2; side++) {
        const int mth = side == 0 ? lo : hi;
        if (mth == 1 || mth == 3) {
            const int kb = side == 0 ? 1 : d.mz;
            const long long cb = cid(d, i, j, kb);
            for (int kbc = 1; kbc <= d.mbc; kbc++) {
                const int kg = side == 0 ? 1 - kbc : d.mz + kbc;
                const long long cg = cid(d, i, j, kg);
                const double sc = zf(side, kbc - 1);   // FP64 factor, one rounding per ghost value
                for (int m = 0; m < 5; m++) q[m * d.P + cg] = (float)((double)q[m * d.P + cb] * sc);
                for (int m = 5; m < nc; m++) q[m * d.P + cg] = q[m * d.P + cb];
            }
            if (mth == 3)
                for (int kbc = 1; kbc <= d.mbc; kbc++) {
                    const int kg = side == 0 ? 1 - kbc : d.mz + kbc;
                    const int km = side == 0 ? kbc : d.mz + 1 - kbc;
                    q[3 * d.P + cid(d, i, j, kg)] = -q[3 * d.P + cid(d, i, j, km)];
                }
        } else if (mth == 2) {
            for (int kbc = 1; kbc <= d.mbc; kbc++)
                for (int m = 0; m < nc; m++) {
                    float *p = q + (long long)m * d.P;
                    if (side == 0) p[cid(d, i, j, kbc - d.mbc)] = p[cid(d, i, j, d.mz - d.mbc + kbc)];
                    else p[cid(d, i, j, d.mz + kbc)] = p[cid(d, i, j, kbc)];
                }
        }
    }
}
template <class G>
__global__ void k32_bc_z(Dims d, float *q, int nc, int lo, int hi, Zr32 zr, G gate)
{
    b32_bc_z(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, q, nc, lo, hi,
             [&](int side, int k) { return zr.s[side][k]; }, gate);
}

// conserved perturbation -> (rho', u, v, w, T') on every cell
// (src3.f90:242-304 with u_bar = 0):
//   T' = T - T_bar = (p' - rho' (gamma-1) E_bar / rho_bar) / (rho R),
//   p' = (gamma-1) (E' - |m|^2 / (2 rho)),  rho = rho_bar + rho'.
//
// The arithmetic of the conversion and of the reassembly below is FP64 (the
// stored values are FP32): T' is a small difference of the pressure and
// density perturbations' background-weighted parts, and E' a sum of such
// parts, whose FP32 rounding the flow carries into the thin upper layers.
// qin, q, keep and the step's increments: as the FP64 form's conversion
// (bc_src.hip)
template <class G>
__device__ __forceinline__ void b32_src_convert(const uint3 BI, Dims d, const float *qin, float *q, float *keep, Col32 col,
                                                const G &gate, const StepParts<float> &sp)
{
    if (!gate.on()) return;
    PADDED_IJK
    const long long P = d.P;
    const bool has = sp.d[0].base != nullptr;
    float v[10];
#pragma unroll
    for (int m = 0; m < 10; m++) v[m] = m < 5 || (has && m < sp.nc) ? qin[m * P + c] : 0.0f;
    if (has) {
        float acc[10];
        step_parts(sp, ip, jp, kk, d.mbc, acc);
#pragma unroll
        for (int m = 0; m < 10; m++) {
            if (m >= 5 && m >= sp.nc) continue;
            if (keep) keep[m * P + c] = v[m];
            v[m] = v[m] + acc[m];
            if (m == 0 || m >= 5) q[m * P + c] = v[m];
        }
    }
    const double rb = col.rho[kk], Eb = col.E[kk], g1 = col.gam[kk] - 1.0, R = col.R[kk];
    const double rp = v[0], rho = rb + rp;
    const double m2 = v[1], m3 = v[2], m4 = v[3], ep = v[4];
    const double irho = 1.0 / rho;
    const double pp = g1 * (ep - 0.5 * (m2 * m2 + m3 * m3 + m4 * m4) * irho);
    q[4 * P + c] = (float)((pp - rp * (g1 * Eb / rb)) * irho / R);
    q[P + c] = (float)(m2 * irho);
    q[2 * P + c] = (float)(m3 * irho);
    q[3 * P + c] = (float)(m4 * irho);
}
template <class G>
__global__ void k32_src_convert(Dims d, const float *qin, float *q, Col32 col, G gate, StepParts<float> sp)
{
    b32_src_convert(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, qin, q, (float *)nullptr, col, gate, sp);
}

// Reassembly, plume forcing and tracer clamp on the interior
// (src3.f90:380-418, 430-445, 514-607, 616-626):
//   m = u rho,  E' = E_bar rho'/rho_bar + T' rho R/(gamma-1) + |m|^2/(2 rho),
// the heating adding dt*heat to T' first.  Positions and the forcing are
// evaluated in FP64.
template <class G>
__device__ __forceinline__ void b32_src_finish(const uint3 BI, Dims d, float *q, const float *t5, int nc, Col32 col, Forcing f, const G &gate)
{
    if (!gate.on()) return;
    gate.forcing(f.t, f.dt, f.tgauss);
    INTERIOR_IJK
    const long long P = d.P;
    const int kk = k + d.mbc - 1;
    const double rb = col.rho[kk], Eb = col.E[kk], g1 = col.gam[kk] - 1.0, R = col.R[kk];
    const double rp = q[c], rho = rb + rp;
    const double m2 = q[P + c] * rho, m3 = q[2 * P + c] * rho;
    double m4 = q[3 * P + c] * rho;
    double tp = t5[c];
    const double xcell = f.xlower + (i - 0.5) * f.dx - f.t * f.vsrcx;
    const double ycell = f.ylower + (j - 0.5) * f.dy;
    const double zcell = f.zlower + (k - 0.5) * f.dz;
    if (f.forcemth == 1) {
        const double gau = exp(-.5 * ((xcell - f.xpos) * (xcell - f.xpos) / (f.xwidth * f.xwidth))) *
                           exp(-.5 * ((ycell - f.ypos) * (ycell - f.ypos) / (f.ywidth * f.ywidth))) *
                           exp(-.5 * ((zcell - f.zpos) * (zcell - f.zpos) / (f.zwidth * f.zwidth))) *
                           exp(-.5 * ((f.t - f.tcenter) * (f.t - f.tcenter) / (f.twidth * f.twidth)));
        const double ffz = sin(f.omega * (f.t - f.tcenter) - f.propx * (xcell - f.xpos) -
                               f.propz * (ycell - f.ypos));
        m4 = m4 + (f.dt * f.amplitude * gau * ffz) * rho;
    } else if (f.forcemth == 3 && !(zcell > 15000.0)) {
        const double g2 = exp(-.5 * ((xcell - f.xpos) * (xcell - f.xpos) / (f.xwidth * f.xwidth))) *
                          exp(-.5 * ((ycell - f.ypos) * (ycell - f.ypos) / (f.ywidth * f.ywidth))) *
                          f.tgauss;
        const double precipw = f.amplitude * g2;
        if (precipw > 0.1) tp = tp + f.dt * sa_heating(precipw, zcell);
    }
    q[P + c] = (float)m2;
    q[2 * P + c] = (float)m3;
    q[3 * P + c] = (float)m4;
    q[4 * P + c] = (float)(Eb * (rp / rb) + tp * rho * R / g1 + 0.5 * (m2 * m2 + m3 * m3 + m4 * m4) / rho);
    for (int m = 5; m < nc; m++) q[m * P + c] = fmaxD(0.0f, fminD(q[m * P + c], 1.0f));
}
template <class G>
__global__ void k32_src_finish(Dims d, float *q, const float *t5, int nc, Col32 col, Forcing f, G gate)
{
    gate.report();
    b32_src_finish(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, q, t5, nc, col, f, gate);
}


// The FP32 form's own bodies for the batched work-list kernels (batch_ops.h)
struct Form32 {
    // po: the operand block in memory (the factors are indexed by layer)
    struct ZScaleC {
        cptr<BatchOps<float>> po;
        __device__ __forceinline__ float operator()(int m, int side, int kbc, float v, long long, long long, long long) const
        {
            return m >= 5 ? v : (float)((double)v * po->zr.s[side][kbc - 1]);
        }
    };
    __device__ static ZScaleC zscale(const BatchOps<float> &, cptr<BatchOps<float>> po) { return {po}; }
    __device__ static void bc_z(uint3 bi, const BatchOps<float> &o, cptr<BatchOps<float>> po, const StepGate &g)
    {
        b32_bc_z(bi, o.d, o.q, o.nc, o.bcz ? o.bc.m[4] : 0, o.bcz ? o.bc.m[5] : 0,
                 [=](int side, int k) { return po->zr.s[side][k]; }, g);
    }
    __device__ static void convert(uint3 bi, const BatchOps<float> &o, const StepGate &g)
    {
        StepParts<float> sp = o.sp;
        if (o.added) sp.d[0].base = nullptr;
        b32_src_convert(bi, o.d, o.q, o.q, o.qold, o.col, g, sp);
    }
    __device__ static void finish(uint3 bi, const BatchOps<float> &o, const StepGate &g)
    {
        b32_src_finish(bi, o.d, o.q, conducted(o, g), o.nc, o.col, o.f, g);
    }
    __device__ static const float *nu(const BatchOps<float> &o) { return o.nu32; }
    __device__ static const float *kap(const BatchOps<float> &o) { return o.kap32; }
};

template <>
const void *batch_op_fn<float>(int op)
{
    switch (op) {
#define MAGIC_OP(X) case X: return reinterpret_cast<const void *>(&k_batch_op<float, X, Form32>);
    MAGIC_OP(OP_BC) MAGIC_OP(OP_BCUVW) MAGIC_OP(OP_BCZ) MAGIC_OP(OP_BACKUP) MAGIC_OP(OP_RESTORE) MAGIC_OP(OP_CONVERT)
    MAGIC_OP(OP_DIFF_CROSS) MAGIC_OP(OP_DIFF) MAGIC_OP(OP_CONDUCT) MAGIC_OP(OP_COPY_T) MAGIC_OP(OP_FINISH)
#undef MAGIC_OP
    default: return nullptr;
    }
}

// instantiations of the single-grid kernels (the batched driver's are
// k_batch_op, above)
template __global__ void k32_bc_z<GridGate>(Dims, float *, int, int, int, Zr32, GridGate);
template __global__ void k32_src_convert<GridGate>(Dims, const float *, float *, Col32, GridGate, StepParts<float>);
template __global__ void k32_src_finish<GridGate>(Dims, float *, const float *, int, Col32, Forcing, GridGate);

// reference AoS q(meqn, i, j, k) (FP64, full state) <-> perturbation planes:
// the background is subtracted / added in FP64, then rounded.
__global__ void k32_aos_to_pert(Dims d, float *q, const double *aos, int nc, const double *bgrho,
                                const double *bgE)
{
    const uint3 BI = {blockIdx.x, blockIdx.y, blockIdx.z};
    PADDED_IJK
    for (int m = 0; m < nc; m++) {
        const double bg = m == 0 ? bgrho[kk] : (m == 4 ? bgE[kk] : 0.0);
        q[(long long)m * d.P + c] = (float)(aos[c * nc + m] - bg);
    }
}

__global__ void k32_pert_to_aos(Dims d, double *aos, const float *q, int nc, const double *bgrho,
                                const double *bgE)
{
    const uint3 BI = {blockIdx.x, blockIdx.y, blockIdx.z};
    PADDED_IJK
    for (int m = 0; m < nc; m++) {
        const double bg = m == 0 ? bgrho[kk] : (m == 4 ? bgE[kk] : 0.0);
        aos[c * nc + m] = bg + (double)q[(long long)m * d.P + c];
    }
}

}  // namespace magic
