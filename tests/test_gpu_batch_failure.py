"""A scenario of a batch that fails in its sweeps ends as the same grid's
magic_claw3 does: with the step's increments in q and the state before the
step in the backup, while the others go on."""
import numpy as np
import pytest

from tests.helpers import perturbed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp32", "fp64"])
@pytest.mark.parametrize("good_steps", [0, 2])   # fails in its first step, or later
def test_failed_scenario_state(form, good_steps):
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64, MAGIC_ERHO, MagicBatch, MagicError, MagicHIP
    fm = FORM_FP32P if form == "fp32" else FORM_FP64
    scen = [perturbed(*dims, [2, 2, 1, 1, 3, 1], seed=n, vel=0.05, visc=1.0)
            for n, dims in enumerate([(12, 10, 8), (9, 11, 7)])]
    b = MagicBatch([s[2] for s in scen], [s[1] for s in scen], [s[3][:, 0, 0, :].copy() for s in scen],
                   [s[4] for s in scen], form=fm)
    c, p, g, aux, q = scen[1]
    d = MagicHIP(g, p, aux, q, form=fm)
    try:
        def run(n, s, t, dt):
            b.start(s, t, t + 1e9, dt, scen[s][0].dtv, scen[s][0].cflv, n, scen[s][0].mthbc)

        def get(backup):
            if backup:
                assert b.L.magic_restore(b.ctx[1]) == 0
                d.restore()
            return b.get_q(1), d.get_q()
        t, dt = 0.0, 50.0                    # the first attempt is rejected
        if good_steps:
            run(good_steps, 0, t, dt)
            run(good_steps, 1, t, dt)
            b.run()
            t, dtv, _ = d.run_steps(c, good_steps, dt0=dt)
            dt = dtv[4]
            assert b.state(1)["t"] == t and b.state(1)["dt"] == dt
        bad = d.get_q()
        m = g.mbc
        bad[m + 3, m + 4, m + 5, 0] = -1.0
        b.set_q(1, bad)
        d.set_q(bad)
        run(3, 0, b.state(0)["t"], b.state(0)["dt"] or dt)
        run(3, 1, t, dt)
        print(f"[failure] {form} after {good_steps}", flush=True)
        b.run()
        assert b.state(1)["status"] == MAGIC_ERHO
        assert b.state(0)["status"] == 0 and b.state(0)["nsteps"] == 3
        with pytest.raises(MagicError):
            d.claw3(t, t + 1e9, [dt] + list(c.dtv[1:]), c.cflv, [3, 0], c.method, c.mthbc)
        for backup in (False, True):
            qb, qd = get(backup)
            np.testing.assert_array_equal(qb, qd)
    finally:
        b.close()
        d.close()
