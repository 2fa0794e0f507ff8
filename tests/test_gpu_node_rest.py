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


def _variant(nelx, nelz):
    return sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)


@pytest.mark.gpu
def test_further_passes_inside_the_node_launch():
    """An upload forgets the thermal history, so that the step after it, not a multiple of
    ifreq_visc, needs a further pass, which fl_node's launch then runs."""
    from tests import oracle_lib as ol
    print("case: 200x40 elements, upload after 3 steps", flush=True)
    gp, st, m = sweep.make_model(_variant(200, 40), abi.PREC_FP64)
    with m:
        m.download()
        ref = st.copy()
        m.step(3)
        m.download()
        m.upload()
        m.therm_stats()
        m.step(4)
        stats = m.therm_stats()
        m.download()
    assert ol.step(gp, ref, 7, cr=True) == 0
    diff = [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
    assert stats[0] == 0 and stats[1] > 0
    assert not diff


@pytest.mark.gpu
@pytest.mark.parametrize("meshes", [[(200, 40), (60, 20), (37, 70)], [(200, 40), (230, 75), (240, 80), (60, 20)]])
def test_further_passes_inside_a_batch(meshes):
    """The same in a batch, after its element update's launch checked the borders; each
    model against itself alone."""
    print("case: batch of %s, upload after 3 steps" % meshes, flush=True)
    alone = []
    for nelx, nelz in meshes:
        gp, st, m = sweep.make_model(_variant(nelx, nelz), abi.PREC_FP64)
        with m:
            m.step(17)
            m.download()
        alone.append(st)
    made = [sweep.make_model(_variant(nelx, nelz), abi.PREC_FP64) for nelx, nelz in meshes]
    models = [x[2] for x in made]
    b = sweep.Batch(models)
    b.step(3)
    b.close()
    for m in models:
        m.download()
        m.upload()
        m.therm_stats()
    b = sweep.Batch(models)
    b.step(14)
    b.close()
    extra = sum(m.therm_stats()[1] for m in models)
    for (gp, st, m), ref in zip(made, alone):
        m.download()
        assert not [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
        m.close()
    assert extra > 0
