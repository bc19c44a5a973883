"""The sweep's wave-strength form against the oracle's step3 where its branches
part: supersonic and transonic flow in every direction (the entropy fix and
the transverse splits' signs), and in subsonic flow as the other tests.  One
step in FP64 stays within the bar of every step3 test, 1e-12 of each
component's largest value."""
import numpy as np
import pytest

from oracle.oracle import COracle
from tests.helpers import perturbed, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wind", [(0, 0, 0), (330, -340, 350), (-700, 650, -800)])
@pytest.mark.parametrize("dims,meqn", [((17, 15, 16), 6), ((31, 9, 14), 5), ((14, 33, 29), 8)])
def test_transonic_step3_vs_oracle(dims, meqn, wind):
    from magic_master_amd.hip import MagicHIP
    mx, my, mz = dims
    c, p, g, aux, q = perturbed(mx, my, mz, [1, 1, 1, 1, 3, 1], seed=mx, vel=40.0, meqn=meqn)
    q[..., 4] -= 0.5 * (q[..., 1] ** 2 + q[..., 2] ** 2 + q[..., 3] ** 2) / q[..., 0]
    for m in range(3):
        q[..., 1 + m] += wind[m] * q[..., 0]
    q[..., 4] += 0.5 * (q[..., 1] ** 2 + q[..., 2] ** 2 + q[..., 3] ** 2) / q[..., 0]
    dt = 0.5
    qo, cfl_o, st = COracle().step3(g, q, aux, dt, p.nspecadv)
    assert st == 0 and cfl_o < 1.0
    print(f"[waves] grid {dims} meqn {meqn} wind {wind} cfl {cfl_o:.3f}", flush=True)
    d = MagicHIP(g, p, aux, q)
    try:
        cfl_g = d.step3(dt)
        qg = d.get_q()
    finally:
        d.close()
    assert abs(cfl_g - cfl_o) <= 1e-12 * cfl_o
    assert rel_err(qg, qo) <= 1e-12
