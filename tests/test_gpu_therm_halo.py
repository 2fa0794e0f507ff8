"""Cells of 25 to 45 m, whose columns couple so strongly (diff dt / dx^2 up to 6e-2) that a
thermal strip takes more than eight halo columns: further passes stay the exception, in
models alone and in a batch, and the result is the correctly rounded oracle's, bit for bit."""
import os

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))
MESHES = [(360, 60), (300, 45), (240, 40), (200, 34)]


def _model(nelx, nelz, precision=abi.PREC_FP64, scale=0.03):
    """The box, its layers and its geotherm made smaller."""
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    p["rxbo"], p["rzbo"] = p["rxbo"] * scale, p["rzbo"] * scale
    for z in p["zones"]:
        z["hc"] = [h * scale for h in z["hc"]]
        z["age_1"] *= scale
    return sweep.make_model(p, precision)


@pytest.mark.gpu
def test_strongly_coupled_columns_bitwise_equal_to_oracle():
    from tests import oracle_lib as ol
    print("case: 360x60 cells of 25 m, 13 steps", flush=True)
    gp, st, m = _model(360, 60)
    with m:
        m.download()
        ref = st.copy()
        m.step(13)
        m.download()
        unproven = m.therm_stats()[0]
    assert ol.step(gp, ref, 13, cr=True) == 0
    assert unproven == 0
    assert not [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [False, True])
def test_few_further_passes_at_strong_coupling(batch):
    n = 200
    print("case: %s cells of 25-45 m, batch %s, %d steps after 40" % (MESHES, batch, n), flush=True)
    models = [_model(nelx, nelz)[2] for nelx, nelz in MESHES]
    b = sweep.Batch(models) if batch else None
    for steps in (40, n):
        for m in models:
            m.therm_stats()
            if not batch:
                m.step(steps)
        if batch:
            b.step(steps)
    if batch:
        b.close()
    stats = [m.therm_stats() for m in models]
    for m in models:
        m.close()
    print("  further passes %s" % [s[1] for s in stats], flush=True)
    assert not any(s[0] for s in stats)
    # (one step in ten at most: every tenth starts from another dt than the one before)
    assert sum(s[1] for s in stats) <= len(models) * n // 10
