"""New starts that are the same in every column, of mesh sizes where some row's sum lies so
near a rounding tie that a value's last bit hangs on the value to its left over many columns:
the thermal step takes as many passes as the serial order's bits need to get there.  Bit for
bit against the correctly rounded oracle, alone and in a batch."""
import os

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))
# (the first two and the last two need more than four passes in one of their first three steps)
MESHES = [(1511, 25), (2042, 26), (60, 20), (3170, 51), (3072, 63)]


def _model(nelx, nelz):
    return sweep.make_model(sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz),
                            abi.PREC_FP64)


def _expected(gp, st, n):
    from tests import oracle_lib as ol
    ref = st.copy()
    assert ol.step(gp, ref, n, cr=True) == 0
    return ref


def _differing(st, ref):
    return [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]


@pytest.mark.gpu
@pytest.mark.parametrize("nelx,nelz", MESHES)
def test_ties_along_a_row_bitwise_equal_to_oracle(nelx, nelz):
    n = 4
    print("case: %dx%d elements, %d steps" % (nelx, nelz, n), flush=True)
    gp, st, m = _model(nelx, nelz)
    with m:
        m.download()
        ref = _expected(gp, st, n)
        m.step(1)
        m.step(n - 1)
        m.download()
        stats = m.therm_stats()
    print("  further passes %d" % stats[1], flush=True)
    assert stats[0] == 0
    assert not _differing(st, ref)


@pytest.mark.gpu
def test_ties_along_a_row_in_a_batch():
    n = 4
    print("case: batch of %s elements, %d steps" % (MESHES, n), flush=True)
    made = [_model(*mesh) for mesh in MESHES]
    refs = []
    for gp, st, m in made:
        m.download()
        refs.append(_expected(gp, st, n))
    with sweep.Batch([m for _, _, m in made]) as b:
        b.step(n)
    stats = [m.therm_stats() for _, _, m in made]
    print("  further passes %s" % [s[1] for s in stats], flush=True)
    assert not any(s[0] for s in stats)
    for (gp, st, m), ref in zip(made, refs):
        m.download()
        assert not _differing(st, ref)
        m.close()
