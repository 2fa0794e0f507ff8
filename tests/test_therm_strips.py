"""The thermal strips (columns marched by one wave, gf_therm.h): their reciprocals against
IEEE division (CPU), and the step at the mesh sizes where the strips can go wrong --
one to three row strips at and next to their limits (64, 65, 116, 117 rows), the smallest
mesh, widths that are no multiple of a strip's -- with both bottom conditions and shear
heating, bit for bit against the correctly rounded oracle (GPU)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))


def test_strip_reciprocals_are_correctly_rounded(tmp_path):
    exe = str(tmp_path / "rcp_check")
    try:
        subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", os.path.join(HERE, "csrc", "rcp_check.c"),
                        "-o", exe, "-lm"], check=True, capture_output=True)
    except (OSError, subprocess.CalledProcessError) as e:  # no C compiler
        pytest.skip("gcc unavailable: %s" % e)
    out = subprocess.run([exe, "10000000"], check=True, capture_output=True, text=True).stdout
    assert [int(v) for v in out.split()] == [0, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("nelx,nelz,option", [
    (2, 2, ""), (3, 4, "flux"), (2, 63, ""), (7, 64, ""), (12, 115, "flux"), (9, 116, ""), (67, 5, ""),
    (61, 21, "shear"), (130, 64, "shear"), (257, 30, ""), (31, 170, "flux")])
def test_strips_at_their_edges_bitwise_equal_to_oracle(nelx, nelz, option):
    from tests import oracle_lib as ol
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    if option == "flux":  # a bottom heat flux in place of the bottom temperature
        p["itemp_bc"], p["bot_bc"] = 2, 0.03
    if option == "shear":
        p["ishearh"] = 1
    n = 12
    print("case: %dx%d elements, %s, %d steps" % (nelx, nelz, option or "plain", n), flush=True)
    sys.stdout.flush()
    gp, st, m = sweep.make_model(p, abi.PREC_FP64)
    with m:
        m.download()
        ref = st.copy()
        m.step(n - 1)
        m.call("fl_therm")  # a thermal call of its own, between steps
        m.download()
        unconv = m.therm_stats()[0]
    assert ol.step(gp, ref, n - 1, cr=True) == 0
    assert ol.call("gfo_fl_therm", gp, ref, cr=True) == 0
    diff = [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
    assert unconv == 0
    assert not diff
