"""Slabs of a grid's sweeps (no GPU): every block that the adding of increments
(parts.h) looks up for a slab's cells, or reads beside them, is one that the
slab sweeps and that lies in its buffer; the slabs' cells are the whole grid."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from magic_master_amd.build import CSRC, HIPCC

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def table(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("slabs") / "libslabs.so")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-shared",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + CSRC, "-o", so,
                    os.path.join(HERE, "slab_geometry.hip")], check=True, stderr=subprocess.DEVNULL)
    L = C.CDLL(so)

    def get(dims, shapes, w, meqn=6):
        out = np.zeros((512, 3, 16), dtype=np.int64)
        n = L.slab_table((C.c_int * 4)(*dims), meqn, (C.c_int * 3)(*shapes), w,
                         out.ctypes.data_as(C.POINTER(C.c_longlong)), 512)
        assert 0 < n <= 512
        return out[:n]
    return get


def _lookups(d, i, n, nA, CI, TA, nt):
    """parts.h:add_parts' blocks along x of cell i: its own and the edge's."""
    if d == 0:
        own = 1 <= i <= n
        x = min(max(i - 1, 0), n - 1)
        lb = x // CI
        return [lb, lb + 1 if own and x % CI == CI - 1 else lb]
    inside = -1 <= i <= nA + 2
    x = min(max(i, -1), nA + 2)
    lb, lo = x // TA, x % TA + 1
    own = inside and x >= 0 and lb < nt
    before, after = x >= 1 and lo == 1, x + 1 <= nA + 1 and lo == TA
    eb = lb - 1 if before else lb + 1
    if lb < 0 or lb >= nt:
        lb = eb
        own = False
    return [lb, eb if inside and (before or after) else lb]


@pytest.mark.parametrize("mx", [1, 2, 3, 13, 14, 15, 16, 17, 28, 29, 30, 31, 46, 47, 48, 62, 63, 64, 97, 124, 130])
@pytest.mark.parametrize("mbc", [2, 3])
def test_blocks_of_a_slab(table, mx, mbc):
    for shapes in [(0, 0, 0), (1, 2, 3), (3, 0, 1), (2, 3, 0)]:
        for w in (0, 16, 32, 48):
            t = table((mx, 11, 9, mbc), shapes, w)
            cells = []
            for slab in t:
                cells += list(range(slab[0][0], slab[0][1]))
                for d in range(3):
                    i0, i1, lo, hi, first, last, nk, nt, ns, CI, TA, n, nA, sT, sK, sS = (int(v) for v in slab[d])
                    assert 0 <= lo < hi <= (nk if d == 0 else nt)
                    if w == 0:
                        assert (lo, hi) == (0, nk if d == 0 else nt)
                    for i in range(i0, i1):
                        for b in _lookups(d, i, n, nA, CI, TA, nt):
                            assert lo <= b < hi, (mx, shapes, w, d, i, b, lo, hi)
                    other = nt if d == 0 else nk
                    numbers = [s * sS + (b * sK + o * sT if d == 0 else o * sK + b * sT)
                               for s in range(ns) for o in range(other) for b in range(lo, hi)]
                    assert sorted(numbers) == list(range(first, last))
            assert cells == list(range(1 - mbc, mx + mbc + 1))
