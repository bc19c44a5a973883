// Declarations shared by the boundary/source kernels and the C ABI.
#pragma once
#include <hip/hip_runtime.h>

namespace magic {

template <typename T>
__device__ __forceinline__ T fminD(T a, T b) { return a < b ? a : b; }
template <typename T>
__device__ __forceinline__ T fmaxD(T a, T b) { return a > b ? a : b; }

struct Dims {
    int mx, my, mz, mbc;
    int NX, NY, NZ;       // padded extents
    long long P;          // NX*NY*NZ
};

// Background planes the source pass reads (aux slots 1-5, 18, 19).
struct Aux {
    const double *rho, *mx, *my, *mz, *E, *R, *gam;
};

// Forcing of src3 (forcemth 1 and 3), evaluated at time t over dt.
struct Forcing {
    int forcemth;
    double t, dt, xlower, ylower, zlower, dx, dy, dz;
    double amplitude, xpos, ypos, zpos, xwidth, ywidth, zwidth, tcenter, twidth;
    double omega, propx, propz, vsrcx;
    double tgauss;        // exp(-.5*((t-tcenter)**2/twidth**2)), host FP64
};

// Gate of the shared kernels for a single grid; kernel arguments are used
// as passed.  Always on, or with scal (the sweeps' Courant number and status
// words) only in a step that the control loop will accept, so that the source
// pass is launched behind the sweeps without waiting for their result; its
// last kernel then hands the words to the host (host: pinned).  With the copy
// and the wait between the two, a step of 12 x 10 x 8 took 83 us (now 79), of 64 x
// 64 x 48 190 us (181).
struct GridGate {
    const unsigned long long *scal = nullptr;
    unsigned long long *host = nullptr;
    double limit = 0.0;
    __device__ __forceinline__ bool on() const
    {
        return !scal || (__longlong_as_double((long long)scal[0]) <= limit && *(const int *)(scal + 1) == 0);
    }
    // by the lanes of one workgroup of the pass's last kernel, on or off
    __device__ __forceinline__ void report() const
    {
        const int t = (int)(threadIdx.y * blockDim.x + threadIdx.x);
        if (host && t < 8 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) host[t] = scal[t];
    }
    template <typename T>
    __device__ __forceinline__ T f(T x, int) const { return x; }
    // whether conduct has a substep kk
    __device__ __forceinline__ bool conducts(int) const { return true; }
    __device__ __forceinline__ void forcing(double &, double &, double &) const {}
};

enum { CLAMP_BC = 1, UVW_BC = 2 };   // modes of the boundary kernel (b_bc)
// Lanes of the boundary kernel: ghost layers, ghost rows of interior layers,
// ghost columns of interior rows, and with the clamp the interior cells,
// CLAMP_LAYERS of a column to a lane (with one each, finding the cell took
// longer than reading it: FP32 batch of 8 grids of 200 x 200 x 300 529 -> 129 us).
constexpr int CLAMP_LAYERS = 8;
__host__ __device__ __forceinline__ unsigned bc_lanes(const Dims &d, int part)
{
    const unsigned g = 2u * d.mbc;
    return part == 0 ? g * d.NX * d.NY : part == 1 ? g * d.NX * d.mz : part == 2 ? g * d.my * d.mz
                                                                                 : (unsigned)d.mx * d.my * ((d.mz + CLAMP_LAYERS - 1) / CLAMP_LAYERS);
}

// bc3's faces (mthbc; 0: skipped)
struct Faces {
    int m[6];
};
// The z pass's scaling (bc3_mpi.f:544-809) of component m's value v of the
// column's boundary cell for its ghost layer kbc: FP64 form with the aux
// planes and the precomputed factors
struct ZScale64 {
    const double *aux1, *aux2, *aux3, *aux5, *zratio;
    int mbc;
    long long NXY;
    __device__ __forceinline__ double operator()(int m, int side, int kbc, double v, long long cg, long long cb,
                                                 long long col) const
    {
        if (m >= 5) return v;
        const double sc = zratio[((long long)side * mbc + (kbc - 1)) * NXY + col];
        if (m == 3) return v * sc;
        const double *a = m == 0 ? aux1 : m == 1 ? aux2 : m == 2 ? aux3 : aux5;
        return a[cg] + (v - a[cb]) * sc;
    }
};

// Stephan & Alexander convective heating profile (src3.f90:534-572) for a
// precipitation rate precipw > 0.1 at height zcell (m): K/s.
__device__ __forceinline__ double sa_heating(double precipw, double zcell)
{
    const double pi = 3.141592653589793;
    const double th = 10.79 + 0.05 * precipw, ph = 6.93 - 0.03 * precipw;
    const double hamp = -0.0001 + 0.0025 * precipw;
    const double tc = 1.12 + 0.10 * precipw, pc = 0.63 + 0.02 * precipw;
    const double bc = 0.37 + 0.00 * precipw, camp = -0.0003 - 0.0005 * precipw;
    const double z2 = zcell / 1000.0;
    double heat;
    if ((bc <= z2) && (z2 <= pc)) heat = camp * sin((2.0 * pi / (4.0 * (pc - bc))) * (z2 - bc));
    else if ((pc <= z2) && (z2 <= tc)) heat = -camp * sin((2.0 * pi / (4.0 * (tc - pc))) * (z2 - tc));
    else if ((pc <= z2) && (z2 <= ph)) heat = hamp * sin((2.0 * pi / (4.0 * (ph - tc))) * (z2 - tc));
    else if ((ph <= z2) && (z2 <= th)) heat = -hamp * sin((2.0 * pi / (4.0 * (th - ph))) * (z2 - th));
    else heat = 0.0;
    return heat;
}

template <class G>
__global__ void k_bc_z(Dims d, double *q, int nc, int lo, int hi, const double *aux1,
                       const double *aux2, const double *aux3, const double *aux5,
                       const double *zratio, G gate);
template <typename T, class ZF, class G>
__global__ void k_bc(Dims d, T *q, int nc, Faces f, int mode, ZF zf, G gate);
template <typename T, class G>
__global__ void k_clamp(T *q, long long P, int nc, G gate);
template <typename T>
struct StepParts;
template <bool COL, class G>
__global__ void k_src_convert(Dims d, const double *qin, double *q, const Aux a, G gate, StepParts<double> sp);
template <typename T, bool COLC, class G>
__global__ void k_diff_cross(Dims d, T *u, const T *q, const T *coef, T dxy, T dxz, T dyz, int kb, G gate);
// y-rows per lane of the directional passes (diff_passes): two load too much
// beside their own (FP32 batch of 8 grids of 200 x 200 x 300: 1.19 ms, four
// 0.78), six leave too few waves (0.96)
constexpr int DIFF_ROWS = 4;
// The operands of the directional passes: diffuse's per velocity component,
// and a substep of conduct.
template <typename T>
struct DiffArgs {
    T *q;                  // component planes; 1..3: velocities, 4: T'
    const T *u;            // cross-term result of the velocities
    T *ut, *qt;            // conduction buffers: substep kk writes ut (odd) or qt (even)
    const T *nu, *kap;
    T f[12];               // dt/dx**2, dt/dy**2, dt/dz**2 of each component in turn, with their factors
    int S;                 // out-of-row z-ghost writes of conduct (mz - mx, or 0)
    int kb;                // layers per workgroup
};

template <typename T, bool COLC, class G>
__global__ void k_diff(Dims d, DiffArgs<T> a, int kk, G gate);
template <typename T, class G>
__global__ void k_copy_interior(Dims d, T *dst, const T *src, int nplanes, G gate);
template <bool COL, class G>
__global__ void k_src_finish(Dims d, double *q, const double *t5, int nc, const Aux a, Forcing f, G gate);
__global__ void k_aos_to_planes(double *planes, const double *aos, long long P, int nc);

// ---- FP32 perturbation form (bc_src32.hip) ----
// Background columns at rest, indexed by k + mbc - 1: rho_bar, E_bar,
// gamma (aux19), R (aux18), and rho_bar, E_bar in FP64.
struct Col32 {
    const double *rho, *E, *gam, *R;   // FP64 columns of rho_bar, E_bar, gamma, R
};
// bc3 z-face factors (rho_bar_ghost/rho_bar_boundary)**0.5 per side and layer
struct Zr32 {
    double s[2][8];
};
// FP32 form: with a background at rest every component's perturbation is
// scaled, in FP64 with one rounding
struct ZScale32 {
    Zr32 zr;
    __device__ __forceinline__ float operator()(int m, int side, int kbc, float v, long long, long long, long long) const
    {
        return m >= 5 ? v : (float)((double)v * zr.s[side][kbc - 1]);
    }
};
template <class G>
__global__ void k32_bc_z(Dims d, float *q, int nc, int lo, int hi, Zr32 zr, G gate);
template <class G>
__global__ void k32_src_convert(Dims d, const float *qin, float *q, Col32 col, G gate, StepParts<float> sp);
template <class G>
__global__ void k32_src_finish(Dims d, float *q, const float *t5, int nc, Col32 col, Forcing f, G gate);
__global__ void k32_aos_to_pert(Dims d, float *q, const double *aos, int nc, const double *bgrho,
                                const double *bgE);
__global__ void k32_pert_to_aos(Dims d, double *aos, const float *q, int nc, const double *bgrho,
                                const double *bgE);
__global__ void k_planes_to_aos(double *aos, const double *planes, long long P, int nc);

}  // namespace magic
