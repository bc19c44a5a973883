"""claw3 against the same step made of single operators (bc3, b4step3, the
backup copy, step3, src3), bit for bit, where claw3 takes another way through
the step than usual."""
import numpy as np
import pytest

from tests.helpers import interior, perturbed

pytestmark = pytest.mark.gpu


def operator_step(d, c, t, dt):
    """One accepted step; returns the dt it took."""
    d.bc3(c.mthbc)
    d.b4step3()
    d.backup()
    while (cfl := d.step3(dt)) > c.cflv[0]:
        dt = min(c.dtv[1], dt * c.cflv[1] / cfl)
        d.restore()
        d.bc3(c.mthbc)
        d.b4step3()
        d.backup()
    d.src3(t, dt, c.mthbc)
    return dt


@pytest.mark.parametrize("form", ["fp32", "fp64"])
@pytest.mark.parametrize("substeps,dt", [(3, 1.0), (40, 1.0), (40, 50.0)])   # few, many; many with a rejected attempt
def test_many_substeps(form, substeps, dt):
    """A source pass too long to be queued before the step is accepted."""
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64, MagicHIP
    c, p, g, aux, q = perturbed(17, 12, 20, [2, 2, 1, 1, 3, 1], seed=9, vel=0.05, visc=1.0)
    d2 = min(g.dx, g.dy, g.dz) ** 2
    aux[..., 10] = 0.75 * (substeps - 0.5) * 0.45 * d2
    aux[..., 11] = 0.2 * aux[..., 10]
    d = MagicHIP(g, p, aux, q, form=FORM_FP32P if form == "fp32" else FORM_FP64)
    try:
        print(f"[substeps] {form} {substeps} dt {dt}", flush=True)
        _, dtv, _, _, log = d.claw3(0.0, -1.0, [dt, c.dtv[1], 0, 0, 0], c.cflv, [1, 0], c.method, c.mthbc)
        assert log.accepted == ([True] if dt == 1.0 else [False, True])
        got = d.get_q()
        d.restore()
        old = d.get_q()
        d.set_q(q)
        assert operator_step(d, c, 0.0, dt) == log.dt[-1]
        np.testing.assert_array_equal(got, d.get_q())
        d.restore()
        np.testing.assert_array_equal(old, d.get_q())
        assert np.isfinite(got[interior(g)]).all()
    finally:
        d.close()


@pytest.mark.parametrize("form", ["fp32", "fp64"])
def test_sweep_overlap_setting_changes_nothing(form):
    """set_sweep_overlap on and off: the same state, dt and t, bit for bit, on
    one grid and in a batch."""
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64, MagicBatch, MagicHIP
    fm = FORM_FP32P if form == "fp32" else FORM_FP64
    c, p, g, aux, q = perturbed(33, 20, 18, [2, 2, 1, 1, 3, 1], seed=3, vel=0.05, visc=1.0)
    out = []
    for on in (True, False):
        d = MagicHIP(g, p, aux, q, form=fm)
        b = MagicBatch([g], [p], [aux[:, 0, 0, :].copy()], [q], form=fm)
        try:
            d.set_sweep_overlap(on)
            b.set_sweep_overlap(on)
            t, dtv, log = d.run_steps(c, 3, dt0=50.0)
            b.start(0, 0.0, 1e9, 50.0, c.dtv, c.cflv, 3, c.mthbc)
            b.run()
            st = b.state(0)
            out += [(t, dtv[4], d.get_q()), (st["t"], st["dt"], b.get_q(0))]
        finally:
            d.close()
            b.close()
    for o in out[1:]:
        assert o[:2] == out[0][:2]
        np.testing.assert_array_equal(o[2], out[0][2])
