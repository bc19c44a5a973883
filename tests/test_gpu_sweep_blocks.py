"""The sweeps' blocks (tile x chunk x segment) and the adding of their
increments, against the oracle's step3 (FP64, the bar of every step3 test:
1e-12 of each component's largest value):
* sizes around the edges of a tile (16 or 8 pencils), of a chunk (14, 30 or
  62 cells) and of a segment, down to one cell;
* the limiters' carried Courant number (rpn3euX.f:563-619) taken from several
  chunks back;
* with room for one direction's increments only, three steps agree with the
  usual ones to 1e-11 (their sums differ by a few roundings a step).
"""
import numpy as np
import pytest

from oracle.oracle import COracle
from tests.helpers import perturbed, rel_err

pytestmark = pytest.mark.gpu


def _step(g, p, aux, q, dt, shapes=(0, 0, 0)):
    from magic_master_amd.hip import MagicHIP
    d = MagicHIP(g, p, aux, q)
    try:
        d.set_tile_shapes(list(shapes))
        cfl = d.step3(dt)
        return cfl, d.get_q()
    finally:
        d.close()


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 2), (13, 14, 15), (14, 15, 28), (16, 13, 14), (29, 30, 31), (15, 17, 63),
                                  (62, 7, 13), (61, 46, 44), (64, 62, 60)])
@pytest.mark.parametrize("shape", [0, 1, 3])
def test_block_edges_vs_oracle(dims, shape):
    c, p, g, aux, q = perturbed(*dims, [1, 1, 1, 1, 3, 1], seed=sum(dims))
    qo, cfl_o, st = COracle().step3(g, q, aux, 2.0, p.nspecadv)
    assert st == 0
    print(f"[blocks] {dims} shape {shape}", flush=True)
    cfl_g, qg = _step(g, p, aux, q, 2.0, (shape,) * 3)
    assert abs(cfl_g - cfl_o) <= 1e-12 * cfl_o
    assert rel_err(qg, qo) <= 1e-12


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("jump", [3, 20])   # cell of the acoustic jump that sets the Courant number
@pytest.mark.parametrize("shape", [0, 2])
def test_carried_courant_number_across_chunks(axis, jump, shape):
    """A uniform wind with a shear ramp in w from cell 60 on: waves 1, 2 and 3
    vanish exactly there (every number is a small dyadic fraction), so the
    shear's limiter takes the Courant number the last acoustic jump left, up to
    four chunks back."""
    n = 90
    dims = (n, 6, 5) if axis == "x" else (6, n, 5)
    c, p, g, aux, q = perturbed(*dims, [1, 1, 1, 1, 3, 1], seed=1, vel=0.0, ntr_values=False)
    K, J, I = q.shape[:3]
    s = np.arange(I)[None, None, :] if axis == "x" else np.arange(J)[None, :, None]
    q[..., 0] = 1.0
    u = 32.0
    w = np.broadcast_to(np.where(s >= 62, (s - 62) * 0.25, 0.0), (K, J, I))
    q[..., 1:4] = 0.0
    q[..., 1 if axis == "x" else 2] = u
    q[..., 3] = w
    e0 = np.broadcast_to(np.where(s >= jump + 2, 262144.0, 262400.0), (K, J, I))
    q[..., 4] = e0 + 0.5 * (u * u + w * w)
    dt = 2.0
    qo, cfl_o, st = COracle().step3(g, q, aux, dt, p.nspecadv)
    assert st == 0
    print(f"[carry] {axis} jump {jump} shape {shape}", flush=True)
    cfl_g, qg = _step(g, p, aux, q, dt, (shape,) * 3)
    assert abs(cfl_g - cfl_o) <= 1e-12 * cfl_o
    assert rel_err(qg, qo) <= 1e-12


def test_room_for_one_direction():
    import ctypes as C
    from magic_master_amd.hip import MagicHIP, load_library
    L = load_library()      # its HIP runtime's own calls, found through its dependencies
    c, p, g, aux, q = perturbed(200, 180, 40, [1, 1, 1, 1, 3, 1], seed=4, vel=0.05, visc=1.0)
    out = []
    for full in (True, False):
        d = MagicHIP(g, p, aux, q)
        fill = C.c_void_p()
        try:
            if not full:   # leave 230 MB: one direction's increments take about 120 MB, all three 350 MB
                free, total = C.c_size_t(), C.c_size_t()
                assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
                assert L.hipMalloc(C.byref(fill), C.c_size_t(free.value - 230_000_000)) == 0
            print(f"[room] full {full}", flush=True)
            d.bc3(c.mthbc)
            d.backup()
            cfl = d.step3(1.0)
            d.restore()
            t, dtv, log = d.run_steps(c, 3, dt0=60.0)    # the first attempt is rejected
            assert not log.accepted[0]
            out.append((cfl, log.dt, d.get_q()))
            d.restore()                                  # the backup holds the last step's start
            out[-1] += (d.get_q(),)
        finally:
            d.close()
            L.hipFree(fill)
    (cfl0, dt0, q0, b0), (cfl1, dt1, q1, b1) = out
    assert cfl0 == cfl1
    np.testing.assert_allclose(dt0, dt1, rtol=1e-13)
    # one step's sums differ by a few roundings; three steps carry them on
    assert rel_err(q1, q0) <= 1e-11 and rel_err(b1, b0) <= 1e-11


def test_report_orders_differ():
    """The error report's two FP64 orders of additions: other last bits, the
    same state to the report's bar (1e-12 of each field's peak)."""
    from magic_master_amd import report
    from magic_master_amd.hip import FORM_FP64
    c, p, g, aux, q = perturbed(40, 20, 18, [1, 1, 1, 1, 3, 1], seed=5, vel=0.3)
    rows = report.compare_runs(c, p, g, aux, q, 20.0, 20.0, (FORM_FP64, True), (FORM_FP64, False))
    worst = [rows[0][k]["max_rel"] for k in ("w", "T'", "rho'")]
    assert max(worst) > 0.0 and max(worst) <= 1e-12, worst
