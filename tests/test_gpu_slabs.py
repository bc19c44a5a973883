"""Little room for the sweeps' increments: a grid swept in slabs, and a batch
swept in several groups, give the same results as with all the room, bit for
bit (every cell's sum is formed whole and in one order)."""
import numpy as np
import pytest

from tests.helpers import perturbed

pytestmark = pytest.mark.gpu


def _form(name):
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64
    return FORM_FP32P if name == "fp32" else FORM_FP64


@pytest.mark.parametrize("form", ["fp32", "fp64"])
@pytest.mark.parametrize("dims,meqn,shapes", [((15, 9, 7), 6, (0, 0, 0)), ((16, 20, 12), 5, (0, 0, 0)), ((33, 17, 20), 6, (1, 2, 3)),
                                              ((100, 6, 5), 10, (0, 0, 0)), ((64, 31, 30), 6, (3, 0, 2)), ((130, 18, 33), 6, (0, 0, 0))])
def test_grid_in_slabs(form, dims, meqn, shapes):
    from magic_master_amd.hip import MagicHIP
    c, p, g, aux, q = perturbed(*dims, [2, 2, 1, 1, 3, 1] if dims[0] > 15 else [1, 1, 1, 1, 3, 1], seed=sum(dims), vel=0.05, visc=1.0, meqn=meqn)
    out = []
    for room in (0, 1):                      # all, the narrowest slabs
        d = MagicHIP(g, p, aux, q, form=_form(form))
        try:
            print(f"[slabs] {form} {dims} room {room}", flush=True)
            d.set_tile_shapes(shapes)
            d.set_increment_room(room)
            d.timing(True)
            d.bc3(c.mthbc)
            d.backup()
            cfl = d.step3(1.0)
            n = d.timing_read()["sweep_x"][1]
            assert n == 1 if room == 0 else n > 1 or dims[0] < 48    # the borders of two slabs hold a small grid
            one = d.get_q()
            d.restore()
            t, dtv, log = d.run_steps(c, 3, dt0=60.0)
            assert not log.accepted[0]
            res = [cfl, one, t, dtv, log.dt, log.cfl, d.get_q()]
            d.restore()
            out.append(res + [d.get_q()])
            d.tune(1.0, reps=1)
            np.testing.assert_array_equal(d.get_q(), out[-1][-1])
        finally:
            d.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("form", ["fp32", "fp64"])
@pytest.mark.parametrize("share", [1.2, 0.7, 1e-6])   # of about what all scenarios' increments take: groups, each grid alone, slabs
def test_batch_with_little_room(form, share):
    """Uneven grids with an empty slot between them, first attempts rejected,
    one grid failing: equal to the grids alone."""
    from magic_master_amd.hip import MagicBatch, MagicError, MagicHIP
    scen = [perturbed(*dims, mthbc, seed=n, vel=0.05, visc=1.0)
            for n, (dims, mthbc) in enumerate([((40, 12, 16), [2, 2, 1, 1, 3, 1]), ((20, 9, 6), [1, 1, 1, 1, 3, 1]),
                                               ((33, 14, 13), [1, 1, 2, 2, 3, 1]), ((70, 10, 20), [1, 1, 1, 1, 3, 1]),
                                               ((12, 10, 8), [2, 2, 2, 2, 3, 1])])]
    bad = scen[4][4]
    bad[6, 7, 8, 0] = -1.0
    b = MagicBatch([s[2] for s in scen], [s[1] for s in scen], [s[3][:, 0, 0, :].copy() for s in scen],
                   [s[4] for s in scen], form=_form(form))
    try:
        b.remove(1)
        el = 4 if form == "fp32" else 8
        total = sum(2.5 * 3 * np.prod(np.array(s[4].shape)) * el for s in scen)     # 4-5 times q, more on small grids
        b.set_increment_room(max(1, int(share * total)))
        for s, (c, p, g, aux, q) in enumerate(scen):
            if s != 1:
                b.start(s, 0.0, 1e9, 60.0, c.dtv, c.cflv, 3, c.mthbc)
        print(f"[room] {form} {share}", flush=True)
        b.run()
        for s, (c, p, g, aux, q) in enumerate(scen):
            if s == 1:
                continue
            st = b.state(s)
            d = MagicHIP(g, p, aux, q, form=_form(form))
            try:
                if s == 4:
                    assert st["status"] == 1
                    with pytest.raises(MagicError):
                        d.claw3(0.0, 1e9, [60.0] + list(c.dtv[1:]), c.cflv, [3, 0], c.method, c.mthbc)
                else:
                    t, dtv, log = d.run_steps(c, 3, dt0=60.0)
                    assert st["status"] == 0 and st["t"] == t and st["dt"] == dtv[4] and st["rejects"] == log.accepted.count(False) > 0
                np.testing.assert_array_equal(b.get_q(s), d.get_q())
                assert b.L.magic_restore(b.ctx[s]) == 0
                d.restore()
                np.testing.assert_array_equal(b.get_q(s), d.get_q())
            finally:
                d.close()
    finally:
        b.close()


def test_no_room_beside_the_grid():
    """A grid whose increments have to go to its staging buffer, with a snapshot
    still on its way out of that buffer."""
    import ctypes as C
    from magic_master_amd.hip import MagicHIP, PinnedBuffer, load_library, snapshot_wait
    L = load_library()      # its HIP runtime's own calls, found through its dependencies
    c, p, g, aux, q = perturbed(400, 150, 100, [1, 1, 1, 1, 3, 1], seed=6, vel=0.05, visc=1.0)
    buf = PinnedBuffer(8 * q.size)
    out = []
    d = MagicHIP(g, p, aux, q)
    fill = C.c_void_p()
    try:
        for full in (True, False):
            if not full:    # leave 100 MB; slabs 16 cells wide take 190 MB beside the grid
                d.set_increment_room(0)
                free, total = C.c_size_t(), C.c_size_t()
                assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
                assert L.hipMalloc(C.byref(fill), C.c_size_t(free.value - 100_000_000)) == 0
            print(f"[no room] full {full}", flush=True)
            d.set_q(q)
            d.timing(True)
            d.timing_reset()
            h = d.snapshot_begin(buf)
            t, dtv, log = d.run_steps(c, 2, dt0=60.0)
            snapshot_wait(h)
            assert full == (d.timing_read()["sweep_x"][1] == len(log.dt))
            out.append([t, log.dt, log.cfl, buf.array(g.shape_q).copy(), d.get_q()])
    finally:
        d.close()
        L.hipFree(fill)
        buf.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(out[0][3], q)
