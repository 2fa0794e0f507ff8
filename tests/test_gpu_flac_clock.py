"""gf_flac and itest_mesh hand their results to the host from the call's last launch: a
loop of gf_flac with the caller's own nloop and time leaves what gf_step leaves, a time
the caller sets comes back unchanged, and the smallest angle does not depend on earlier
calls.  Meshes of one workgroup of elements, of exactly two, of one element more, and of 64
workgroups (up to which that launch hands over itself) and 65."""
import os

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
@pytest.mark.parametrize("nelx,nelz,precision", [
    (2, 2, abi.PREC_FP64), (32, 16, abi.PREC_FP64), (19, 27, abi.PREC_FP64), (60, 20, abi.PREC_MIXED),
    (128, 128, abi.PREC_FP64), (129, 128, abi.PREC_FP64)])
def test_flac_loop_equals_step(nelx, nelz, precision):
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    print("case: %dx%d elements, precision %d" % (nelx, nelz, precision), flush=True)
    gp, st, m = sweep.make_model(p, precision)
    gp2, st2, m2 = sweep.make_model(p, precision)
    with m, m2:
        c = st.clock
        angles = []
        for _ in range(13):
            m.call("flac")
            c.nloop += 1
            c.time += c.dt
            angles.append(m.itest_mesh(3, 1.3, 11.0))
        m2.step(13)
        assert m2.itest_mesh(3, 1.3, 11.0) == angles[-1] == m.itest_mesh(3, 1.3, 11.0)
        for f in ("nloop", "nsrate", "time", "dt", "dtavg", "dt_elastic", "dt_maxwell"):
            assert getattr(st.clock, f) == getattr(st2.clock, f), f
        m.download()
        m2.download()
        c.time = 3.25e15
        m.call("flac")
        assert c.time == 3.25e15
    diff = [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(st2, f))]
    assert not diff
