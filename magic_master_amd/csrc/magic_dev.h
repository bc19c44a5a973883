// Shared declarations of the MAGIC device kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace magic {

// A compile-time int passed as a value (to generic lambdas).
template <int V>
struct IConst { static constexpr int value = V; };

// One directional sweep of step3 (lib/step3.f:121-621): pencils along the
// normal direction n, with the "g" transverse direction (gadd, flux3fw.f:419)
// and the "h" transverse direction (hadd, flux3fw.f:545).
//   x-sweep: n = x, g = y, h = z      y-sweep: n = y, g = z, h = x
//   z-sweep: n = z, g = x, h = y      (step3.f:161, 329, 499 argument order)
template <typename T>
struct SweepArgsT {
    const T *__restrict__ qold;        // component planes, stride P
    T *__restrict__ qnew;
    const double *__restrict__ gam;    // aux(19) plane
    const double *__restrict__ vgrav;  // aux(17) plane
    long long P;                       // cells per plane
    int comp[10];                      // local component -> plane (rho, m_n, m_g', m_h', E, tracers)
    int n;                             // interior cells along the pencil
    int nA, nB;                        // interior extents along g and h
    int mbc;
    long long sN, sA, sB;              // strides (cells) along n, g, h
    int cA, cB;                        // pencil colour (a mod 3, b mod 3)
    int gravity;                       // 1 on the z-sweep (rpn3euX.f:202-208)
    int nspecadv;
    int sweep;                         // 1, 2, 3 (for error reports)
    double dtdn, fg, fh;               // dt/dn, dt/dg, dt/dh
    unsigned long long *cfl_bits;      // running max of the Courant number
    int *status;                       // [0] code, [1..4] sweep,i,j,k of first failure
    // perturbation form only: background columns indexed by k + mbc - 1
    // (rho_bar, E_bar, gamma, aux17, and the background's own z jump
    // p_bar(k) - p_bar(k-1) - .5 (rho_bar(k) + rho_bar(k-1)) aux17(k))
    const double *crho, *cE, *cgam, *cvg, *cres;
    // tiled sweep: sA/sB/nA/nB then describe the tile axis a and the marching
    // axis b; a_is_g: the tile axis is the sweep's g direction
    int a_is_g;
    long long cofs[10];                // cells to the planes of rho, the momenta along n, a and b, E, tracers
    T *parts;                          // the direction's increment blocks (SweepParts)
    int lgL, sT, sK, sS;               // log2 planes per segment; blocks between tiles, chunks, segments
};
using SweepArgs = SweepArgsT<double>;

template <int NTR>
__global__ void sweep_kernel(SweepArgs a);

// Tiled sweep, one instantiation per tile shape SH (0 .. TILE_NSHAPE-1):
// a workgroup sweeps TA = tile_ta(SH) pencils along the tile axis a by 256/TA
// interfaces along the pencils, over a segment of planes along b, and writes
// the increments of its block to the block's part.  (T, PERT) = (double,
// false): FP64 form; (float, true): FP32 perturbation form.  items: {argument
// block, tile, chunk, segment} of each workgroup; run[argument block] points
// at the grid's "runs in this attempt" flag.
constexpr int TILE_NSHAPE = 4;
__host__ __device__ constexpr int tile_ta(int sh) { return sh == 0 ? 16 : sh == 3 ? 4 : 8; }
__host__ __device__ constexpr int tile_lgta(int sh) { return sh == 0 ? 4 : sh == 3 ? 2 : 3; }
// cells along the pencil a chunk completes, and positions of a part's plane
__host__ __device__ constexpr int tile_ci(int sh) { return 256 / tile_ta(sh) - 2; }
__host__ __device__ constexpr int part_npos(int sh) { return (tile_ta(sh) + 2) * (tile_ci(sh) + 1); }
template <typename T, bool PERT, int NTR, int SH>
__global__ void tile_sweep(const SweepArgsT<T> *args, const int4 *items, const int *const *run);

// The increment blocks of one sweep direction.  Block (segment s, chunk k,
// tile t) is number s sS + k sK + t sT, of (L+2) * nc * npos elements: planes
// b = s L - 1 .. s L + L, of each plane nc components (tile order: rho, m_n,
// m_a, m_b, E, tracers) of npos positions (a offsets t TA - 1 .. t TA + TA by
// cells k CI .. k CI + CI).  A cell's increments are its own block's entry
// and, next to a block's edge, the neighbouring blocks' entries for it.
// Whatever the tile's lane order, positions and blocks run fastest along x
// (the pencils of the x-sweep, the tile axis of the others), as the lanes
// that add them to q do.
template <typename T>
struct SweepParts {
    const T *base;         // block 0 (not in the buffer where a slab starts further on); nullptr: no increments pending
    int n, nA, nB;         // interior cells along the pencils, a and b
    int lgTA, lgL;         // log2 pencils per tile, planes per segment
    int CI;                // cells a chunk completes
    unsigned iCI;          // ceil(2**32 / CI)
    int nt, nk, ns;        // tiles, chunks, segments
    int sT, sK, sS;        // blocks between neighbouring tiles, chunks, segments
};

}  // namespace magic
