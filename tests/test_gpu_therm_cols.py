"""The thermal step's two forms (gf_therm.h): a workgroup a strip where every strip has a
CU of its own, marching waves otherwise.  Meshes at and next to the 256 strips where the
form changes, marched meshes whose width is no multiple of a strip's, and columns that
couple so strongly that a mesh changes form once its time step is known; bit for bit
against the correctly rounded oracle."""
import os

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
@pytest.mark.parametrize("nelx,nelz,option", [
    (1023, 8, ""), (1024, 8, "flux"), (1027, 64, "shear"), (510, 115, ""), (513, 116, "flux"), (601, 190, ""),
    (90, 40, "coupled"), (200, 70, "coupled")])
def test_both_forms_bitwise_equal_to_oracle(nelx, nelz, option):
    from tests import oracle_lib as ol
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    if option == "flux":
        p["itemp_bc"], p["bot_bc"] = 2, 0.03
    if option == "shear":
        p["ishearh"] = 1
    if option == "coupled":
        for ph in p["phases"]:
            ph["conduct"] = 40.0 * ph["conduct"]
    print("case: %dx%d elements, %s" % (nelx, nelz, option or "plain"), flush=True)
    gp, st, m = sweep.make_model(p, abi.PREC_FP64)
    with m:
        m.download()
        ref = st.copy()
        m.step(2)
        m.step(9)
        m.call("fl_therm")
        m.download()
        unconv = m.therm_stats()[0]
    assert ol.step(gp, ref, 11, cr=True) == 0
    assert ol.call("gfo_fl_therm", gp, ref, cr=True) == 0
    diff = [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
    assert unconv == 0
    assert not diff
