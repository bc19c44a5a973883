"""The one-pass boundary kernel and the fused source-pass passes against the
oracle (bc3 and src3 as sequential passes):
* bc3 with every mixture of extrapolating, periodic, wall and skipped faces,
  down to two cells per axis: every ghost cell as the three passes leave it
  (only the z faces round: 1e-14 of each component's largest value, the bar
  of the bc3 tests);
* src3 with several diffusion and conduction substeps where conduct's z ghosts
  stop short of a row (mx > mz), cross into the next layer's ghost rows, and
  reach its interior (mz > 2 mx + 4): 1e-12, the bar of the src3 tests.
"""
import itertools

import numpy as np
import pytest

from oracle.oracle import COracle
from tests.helpers import interior, perturbed, rel_err

pytestmark = pytest.mark.gpu

DT = 5.6   # s, about what the perturbed grids settle at


@pytest.mark.parametrize("dims,meqn", [((7, 6, 5), 7), ((2, 3, 4), 5), ((65, 3, 2), 6)])
@pytest.mark.parametrize("form", ["fp64", "fp32"])
def test_mixed_faces(dims, meqn, form):
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64, MagicHIP
    c, p, g, aux, q = perturbed(*dims, [1] * 6, seed=3, meqn=meqn)
    tol = 1e-14
    if form == "fp32":   # the ghost perturbations round once more in FP32
        tol = 1e-7
    O = COracle()
    d = MagicHIP(g, p, aux, q, form=FORM_FP32P if form == "fp32" else FORM_FP64)
    try:
        for n, xy in enumerate(itertools.product([1, 2, 3, -1], repeat=4)):
            faces = list(xy) + [[1, 3], [3, 1], [-1, 3], [1, -1], [-1, -1]][n % 5]
            d.set_q(q)
            qo = d.get_q()
            assert O.bc3(g, qo, aux, faces) == 0
            d.bc3(faces)
            assert rel_err(d.get_q(), qo) <= tol, faces
    finally:
        d.close()


@pytest.mark.parametrize("dims", [(20, 9, 6), (6, 5, 13), (4, 7, 15), (5, 9, 40), (66, 6, 37)])
def test_src3_substeps(dims):
    from magic_master_amd.hip import MagicHIP
    c, p, g, aux, q = perturbed(*dims, [1, 1, 2, 2, 3, 1], seed=sum(dims), visc=1e6)
    top = aux[g.mz + g.mbc - 1, g.mbc, g.mbc].copy()     # scale so that 3 diffusion substeps of 2 conduction substeps run
    d2 = min(g.dx, g.dy, g.dz) ** 2
    aux[..., 10] *= 2.5 * 0.45 * d2 / 5.0 / (4.0 / 3.0 * top[10])
    aux[..., 11] *= 1.5 * 0.45 * d2 / (5.0 / 3.0) / top[11]
    p.tcenter = 0.0
    qo = q.copy()
    st, ndtr_o, ndtrc_o = COracle().src3(g, p, qo, aux, 0.0, 5.0, c.mthbc)
    assert st == 0 and (ndtr_o, ndtrc_o) == (3, 2)
    d = MagicHIP(g, p, aux, q)
    try:
        assert d.src3(0.0, 5.0, c.mthbc) == (3, 2)
        assert rel_err(d.get_q(), qo, interior(g)) <= 1e-12
    finally:
        d.close()


@pytest.mark.parametrize("form", ["fp32", "fp64"])
def test_batch_substeps(form):
    """A batch of grids with two diffusion substeps of two conduction substeps
    each (and one grid with one of each) equals the grids run alone, bitwise."""
    from tests.test_gpu_batch import _batch, _single
    scen = []
    for n, (dims, mthbc, more) in enumerate([((6, 5, 13), [1, 1, 2, 2, 3, 1], True), ((20, 9, 6), [2, 2, 1, 1, 3, 1], True),
                                             ((5, 9, 40), [1, 1, 1, 1, 3, 1], True), ((12, 10, 8), [2, 2, 2, 2, 3, 1], False)]):
        c, p, g, aux, q = perturbed(*dims, mthbc, seed=20 + n, visc=1e6, vel=0.05)
        p.tcenter = 1e9
        top = aux[g.mz + g.mbc - 1, g.mbc, g.mbc].copy()
        d2 = min(g.dx, g.dy, g.dz) ** 2
        for slot, want, dt in [(10, 1.9, 4.0 / 3.0 * DT), (11, 1.9, DT / 2.0)]:
            aux[..., slot] *= (want if more else 0.5) * 0.45 * d2 / dt / top[slot]
        scen.append((c, p, g, aux, aux[:, 0, 0, :].copy(), q))
    states, qb = _batch(scen, 4, DT, form=form)
    for k, (c, p, g, aux, col, q) in enumerate(scen):
        t, dt_next, qs, log = _single(c, p, g, aux, q, c.mthbc, 4, DT, form=form)
        assert states[k]["status"] == 0 and states[k]["nsteps"] == 4
        top = aux[g.mz + g.mbc - 1, g.mbc, g.mbc]
        d2 = min(g.dx, g.dy, g.dz) ** 2
        counts = set()
        for dt, ok in log:
            n1 = int(np.ceil(dt * 4.0 / 3.0 * top[10] / d2 / 0.45))
            counts.add((n1, int(np.ceil(dt / n1 * top[11] / d2 / 0.45))))
        assert (max(counts) >= (2, 2)) == (k < 3), counts
        assert states[k]["t"] == t and states[k]["dt"] == dt_next
        np.testing.assert_array_equal(qb[k], qs)


@pytest.mark.parametrize("form", ["fp32", "fp64"])
@pytest.mark.parametrize("dt", [0.5, 50.0])   # accepted, and rejected once before
def test_claw3_refused_source(form, dt):
    """A source pass that src3 refuses (a wind that changes with time) ends
    claw3 with its error after the accepted sweeps: q holds their increments."""
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64, MagicError, MagicHIP
    c, p, g, aux, q = perturbed(17, 12, 20, [2, 2, 1, 1, 3, 1], seed=5, vel=0.05)
    p.omega1 = 1.0
    d = MagicHIP(g, p, aux, q, form=FORM_FP32P if form == "fp32" else FORM_FP64)
    try:
        with pytest.raises(MagicError):
            d.claw3(0.0, -1.0, [dt, c.dtv[1], 0, 0, 0], c.cflv, [1, 0], c.method, c.mthbc)
        got = d.get_q()
        d.set_q(q)
        d.bc3(c.mthbc)
        d.b4step3()
        d.backup()
        while (cfl := d.step3(dt)) > c.cflv[0]:
            dt = min(c.dtv[1], dt * c.cflv[1] / cfl)
            d.restore()
            d.bc3(c.mthbc)
            d.b4step3()
            d.backup()
        np.testing.assert_array_equal(got, d.get_q())
    finally:
        d.close()
