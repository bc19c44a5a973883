// The library's slab geometry (ctx.h) for tests/test_slabs.py, on the host.
#include "../magic_master_amd/csrc/ctx.h"

// slabs w cells wide of a grid (dims mx, my, mz, mbc): per slab and direction
// {i0, i1, lo, hi, first block, last block + 1, nk, nt, ns, CI, TA, n, nA, sT, sK, sS}, the
// blocks numbered in the buffer; returns the slabs
extern "C" int slab_table(const int *dims, int meqn, const int *sh, int w, long long *out, int maxslab)
{
    magic_ctx c;
    c.mx = dims[0]; c.my = dims[1]; c.mz = dims[2]; c.mbc = dims[3]; c.meqn = meqn;
    c.d.mx = c.mx; c.d.my = c.my; c.d.mz = c.mz; c.d.mbc = c.mbc;
    c.d.NX = c.mx + 2 * c.mbc; c.d.NY = c.my + 2 * c.mbc; c.d.NZ = c.mz + 2 * c.mbc;
    c.P = c.d.P = (long long)c.d.NX * c.d.NY * c.d.NZ;
    size_t bytes;
    const std::vector<Slab> slabs = Slabs<double>(&c, sh).cut(w ? w : c.mx + 2, bytes);
    long long *o = out;
    for (size_t s = 0; s < slabs.size() && (int)s < maxslab; s++) {
        double *const buf = (double *)(size_t(1) << 40), *next = buf;
        for (int dir = 0; dir < 3; dir++) {
            SweepArgsT<double> a;
            SweepParts<double> p;
            sweep_geometry(&c, dir, sh[dir], a, p);
            double *const from = next;
            const long long bs = block_size(p, meqn, sh[dir]);
            next = parts_layout(a, p, dir, slabs[s].lo[dir], slabs[s].hi[dir], meqn, sh[dir], next);
            const long long v[] = {slabs[s].i0, slabs[s].i1, slabs[s].lo[dir], slabs[s].hi[dir], (from - a.parts) / bs,
                                   (next - a.parts) / bs, p.nk, p.nt, p.ns, p.CI, 1 << p.lgTA, p.n, p.nA, a.sT, a.sK, a.sS};
            memcpy(o, v, sizeof(v));
            o += 16;
        }
        if ((size_t)(next - buf) * sizeof(double) > bytes) return -1;
    }
    return (int)slabs.size();
}
