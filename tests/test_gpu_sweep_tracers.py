"""The sweeps with several tracers against the oracle's step3, for every tile
shape and form: from two tracers on they follow the other components' targets,
and from four on the FP64 form keeps its jumps in the plane of the tile that
is cleared for the next increments.  The grid has two chunks along every axis
for every shape but the widest, and more than one segment, with a remainder in
each.  The bars are those of the step3 tests: 1e-12 in FP64, the FP32 form's
own for its interior perturbations.
"""
import numpy as np
import pytest

from magic_master_amd.report import form_error
from oracle.oracle import COracle
from tests.helpers import perturbed, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("meqn", [7, 8, 9, 10])
def test_tracers_step3_vs_oracle(meqn, shape):
    from magic_master_amd.hip import FORM_FP32P, FORM_FP64, MagicHIP
    c, p, g, aux, q = perturbed(35, 33, 37, [1, 1, 1, 1, 3, 1], seed=meqn, vel=20.0, meqn=meqn)
    qo, cfl_o, st = COracle().step3(g, q, aux, 0.5, p.nspecadv)
    assert st == 0 and cfl_o < 1.0
    for form in (FORM_FP64, FORM_FP32P):
        d = MagicHIP(g, p, aux, q, form=form)
        try:
            d.set_tile_shapes([shape] * 3)
            cfl_g = d.step3(0.5)
            qg = d.get_q()
        finally:
            d.close()
        if form == FORM_FP64:
            assert abs(cfl_g - cfl_o) <= 1e-12 * cfl_o
            assert rel_err(qg, qo) <= 1e-12
        else:
            err = form_error(g, qg, qo, aux)
            assert all(e["max_rel"] <= 1e-5 for e in err.values()), err
