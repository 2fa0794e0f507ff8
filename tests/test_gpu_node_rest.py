"""The end of a thermal call inside fl_node's launch (k_node_rest), on meshes at and next
to the number of tiles up to which it runs there, with a first call that needs a further
pass (200x40 cells, taller than wide) and with a bottom row that fl_node reads; bit for bit
against the correctly rounded oracle."""
import os

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))


# 64 x 4 nodes a tile, at most 768: 3071 x 63 cells have 768 tiles, 3075 x 63 have 769
@pytest.mark.gpu
@pytest.mark.parametrize("nelx,nelz,option,extra", [
    (200, 40, "", True), (200, 40, "flux", True), (3071, 63, "", False), (3075, 63, "", False), (40, 12, "flux", False),
    (200, 40, "sides", True)])
def test_thermal_end_with_the_node_update(nelx, nelz, option, extra):
    from tests import oracle_lib as ol
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    if option == "flux":
        p["itemp_bc"], p["bot_bc"] = 2, 0.03
    if option == "sides":  # hydrostatic side walls, whose densities read the step's temperature
        p["nystressbc"], p["nydrsides"] = 1, 1
        p["bcs"] = [b for b in p["bcs"] if b["nofside"] in (1, 3)]
        p["nofbc"] = len(p["bcs"])
    print("case: %dx%d elements, %s" % (nelx, nelz, option or "plain"), flush=True)
    gp, st, m = sweep.make_model(p, abi.PREC_FP64)
    with m:
        m.download()
        ref = st.copy()
        m.step(7)  # (nothing is left to launches of their own but on multiples of ifreq_visc)
        m.call("fl_therm")
        m.step(6)
        m.download()
        stats = m.therm_stats()
    assert ol.step(gp, ref, 7, cr=True) == 0
    assert ol.call("gfo_fl_therm", gp, ref, cr=True) == 0
    assert ol.step(gp, ref, 6, cr=True) == 0
    diff = [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
    assert stats[0] == 0
    assert not extra or stats[1] > 0
    assert not diff
