"""The library's host code where a run on the GPU cannot reach it: launches
that fail half way, steps rejected by any factor, device memory that runs out.
The library runs with a HIP runtime without a device (tests/hip_stub.cpp,
preloaded into a process of its own): kernels do nothing, so no result of a
step is checked here, only what the host decides."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """Runs a script with the stub; `stub` and the test inputs are in scope."""
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                    os.path.join(ROOT, "tests", "hip_stub.cpp")], check=True)
    head = f"""
import ctypes as C
import numpy as np
from magic_master_amd import problem as P
from magic_master_amd.hip import *
from tests.helpers import perturbed
stub = C.CDLL({so!r})
stub.stub_launches.restype = C.c_char_p
stub.stub_used.restype = C.c_size_t
stub.stub_room.argtypes = [C.c_size_t]
def courant(*c):
    stub.stub_courant((C.c_double * len(c))(*c), len(c))
def launches():
    out = [l.split()[0] for l in stub.stub_launches().decode().splitlines()]
    stub.stub_clear()
    return out
"""

    def run(script):
        preload = " ".join(filter(None, [so, os.environ.get("LD_PRELOAD")]))
        env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=ROOT)
        r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(script)], env=env, cwd=ROOT,
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
        assert r.returncode == 0, r.stdout
    return run


@pytest.mark.parametrize("substeps", [1, 40])
@pytest.mark.parametrize("cfl", [0.5, 1.9])   # the attempt would be accepted, or rejected
def test_claw3_launch_failure_in_the_source_pass(host, cfl, substeps):
    """A launch that fails behind the source pass's conversion ends claw3 with
    an error, on the state before the step (not on the older backup).  A long
    source pass is launched only once its attempt is accepted."""
    host(f"""
    c, p, g, aux, q = perturbed(8, 7, 6, [1, 1, 1, 1, 3, 1])
    aux[..., 10] = 0.75 * ({substeps} - 0.5) * 0.45 * min(g.dx, g.dy, g.dz) ** 2 / c.dtv[0]
    d = MagicHIP(g, p, aux, q)
    courant(0.5, {cfl}, 0.5)
    one = lambda: d.claw3(0.0, -1.0, c.dtv, c.cflv, [10, 0], c.method, c.mthbc)
    one()
    assert np.all(d.get_q()[..., :5] == 1.0)      # the first step's source pass wrote its mark
    stub.stub_fail(b"6k_diffI", 0)
    try:
        one()
        raise SystemExit("no error")
    except MagicError as e:
        assert e.code == 6, e
    assert np.all(d.get_q()[..., :5] == 1.0), d.get_q()[0, 0, 0]
    d.restore()
    assert np.all(d.get_q()[..., :5] == 1.0)
    """)


@pytest.mark.parametrize("dt,rejected", [(1e5, True), (1e30, True), (1e5, False), (2.0, False)])
def test_rejected_attempt_launches_no_substeps(host, dt, rejected):
    """The diffusion substeps an attempt would need grow with its dt (here 999
    at 1e5 s): an attempt that is rejected launches none of them, one that is
    accepted all."""
    host(f"""
    dt, rejected = float("{dt}"), {rejected}
    c, p, g, aux, q = perturbed(8, 7, 6, [1, 1, 1, 1, 3, 1], visc=1.0)
    d2 = min(g.dx, g.dy, g.dz) ** 2
    aux[..., 10] = aux[..., 11] = 1e3 * 0.45 * d2 / 1e5 * 0.75 * 0.999
    d = MagicHIP(g, p, aux, q)
    courant(*[1e4, 0.5] if rejected else [0.5])
    d.claw3(0.0, -1.0, [dt, 1.0, 0, 0, 0], c.cflv, [10, 0], c.method, c.mthbc)
    n = sum("k_diff_cross" in l for l in launches())
    if rejected:
        assert n == 1, n                  # those of the second attempt (dt 1)
    else:
        assert n == (999 if dt > 10 else 1), n
    """)


@pytest.mark.parametrize("fails", [0, 7])   # the first candidate, a later one
def test_tune_failure_restores_the_backup(host, fails):
    """A tuner that ends with an error leaves the backup a copy of q, its ghost
    cells among them."""
    host(f"""
    c, p, g, aux, q = perturbed(8, 7, 6, [1, 1, 1, 1, 3, 1])
    d = MagicHIP(g, p, aux, q)
    launches()
    stub.stub_fail(b"tile_sweep", {fails})
    try:
        d.tune(1.0)
        raise SystemExit("no error")
    except MagicError:
        pass
    l = launches()
    assert any("4k_bc" in n for n in l) and "copy" in l[[i for i, n in enumerate(l) if "4k_bc" in n][-1]:], l
    assert d.tile_shapes() == [0, 0, 0]
    """)


@pytest.mark.parametrize("fails", [-1, 0, 7])   # none, the first candidate, a later one
def test_batch_tune_restores_the_backups(host, fails):
    """The batch's tuner leaves every scenario's backup a copy of its q, ghost
    cells among them, whether it succeeds or not."""
    host(f"""
    b = MagicBatch([], [], [], meqn=6, mbc=2, maux=32, form=FORM_FP64)
    for n in range(3):
        c, p, g, aux, q = perturbed(8 + n, 7, 6, [1, 1, 1, 1, 3, 1])
        b.add(g, p, aux[:, 0, 0, :].copy(), q)
    launches()
    stub.stub_fail(b"tile_sweep", {fails})
    try:
        b.tune()
        assert {fails} < 0
    except MagicError:
        assert {fails} >= 0
    l = launches()
    last = [i for i, n in enumerate(l) if "4k_bc" in n][-1]
    assert l[last:].count("copy") == 3, l[last:]
    """)


def test_batch_room_found_again(host):
    """A batch that once had room for a part of a grid's increments only goes
    the usual way again once what it holds fits."""
    host("""
    def add(dims):
        c, p, g, aux, q = perturbed(*dims, [1, 1, 1, 1, 3, 1])
        s = b.add(g, p, aux[:, 0, 0, :].copy(), q)
        b.start(s, 0.0, 1e9, 1.0, c.dtv, c.cflv, 5, c.mthbc)
        return s
    backup = lambda: any("k_batch_opIdLi3E" in n for n in launches())
    for share in np.linspace(8.0, 0.5, 30):      # of the big grid's q
        b = MagicBatch([], [], [], meqn=6, mbc=2, maux=32, form=FORM_FP64)
        big = add((60, 50, 40))
        small = add((10, 9, 8))
        launches()
        stub.stub_room(stub.stub_used() + int(share * 64 * 54 * 44 * 48))
        b.run(1, 1)
        if backup():
            break
        b.close()
        stub.stub_room(1 << 60)
    else:
        raise SystemExit("never out of room")
    b.remove(big)
    b.run(1, 1)
    assert not backup()
    """)


def test_no_room_beside_the_grid(host):
    """A grid that fills the device is stepped all the same (its increments go
    to the staging buffer), and a snapshot that is still being copied out of
    that buffer is waited for."""
    host("""
    c, p, g, aux, q = perturbed(400, 30, 30, [1, 1, 1, 1, 3, 1])
    d = MagicHIP(g, p, aux, q)
    stub.stub_room(stub.stub_used() + (1 << 20))        # 6.5 MB are the least beside it
    d.step3(1.0)
    launches()
    buf = PinnedBuffer(8 * q.size)
    h = d.snapshot_begin(buf)
    d.run_steps(c, 2)
    l = launches()
    first = [i for i, n in enumerate(l) if "tile_sweep" in n][0]
    assert "wait" in l[:first][l.index("wait") + 1:], l[:first]   # beside the copy stream's own
    snapshot_wait(h)
    d.close()
    stub.stub_room(1 << 60)
    b = MagicBatch([g], [p], [aux[:, 0, 0, :].copy()], [q], form=FORM_FP64)
    stub.stub_room(stub.stub_used() + (1 << 20))
    b.start(0, 0.0, 1e9, 1.0, c.dtv, c.cflv, 5, c.mthbc)
    b.run(1, 1)
    assert b.state(0)["status"] == 0
    launches()
    h = b.snapshot_begin(0, buf)
    b.run(1, 1)
    assert launches().count("wait") == 2
    snapshot_wait(h)
    b.remove(0)
    stub.stub_room(1 << 60)
    s = b.add(g, p, aux[:, 0, 0, :].copy(), q)
    b.start(s, 0.0, 1e9, 1.0, c.dtv, c.cflv, 5, c.mthbc)
    b.run(1, 1)
    b.close()
    """)


@pytest.mark.parametrize("batch", [False, True])
def test_lists_without_room(host, batch):
    """Where the blocks' lists find no room the call ends with MAGIC_ENOMEM,
    and the next one, with room again, goes on."""
    host(f"""
    c, p, g, aux, q = perturbed(60, 30, 30, [1, 1, 1, 1, 3, 1])
    def grid():
        if not {batch}:
            d = MagicHIP(g, p, aux, q)
            return d, lambda: d.step3(1.0)
        b = MagicBatch([g], [p], [aux[:, 0, 0, :].copy()], [q], form=FORM_FP64)
        b.start(0, 0.0, 1e9, 1.0, c.dtv, c.cflv, 5, c.mthbc)
        return b, lambda: b.run(1, 1)
    d, step = grid()
    before = stub.stub_used()
    step()
    whole = stub.stub_used() - before
    d.close()
    for miss in (1 << 9, 1 << 12):           # the lists take 20 KB, the last allocation of all
        d, step = grid()
        stub.stub_room(stub.stub_used() + whole - miss)
        try:
            step()
            raise SystemExit("no error")
        except MagicError as e:
            assert e.code == 7, e
        stub.stub_room(1 << 60)
        step()
        d.close()
    """)


def test_sweep_overlap_setting_keeps_the_graph(host):
    """The setting that has no effect does not make a batch capture again."""
    host("""
    c, p, g, aux, q = perturbed(12, 10, 8, [1, 1, 1, 1, 3, 1])
    b = MagicBatch([g], [p], [aux[:, 0, 0, :].copy()], [q], form=FORM_FP64)
    b.start(0, 0.0, 1e9, 1.0, c.dtv, c.cflv, 5, c.mthbc)
    b.run(1, 1)
    assert launches()
    for on in (True, False):
        b.set_sweep_overlap(on)
        b.run(1, 1)
        assert not launches()
    """)
