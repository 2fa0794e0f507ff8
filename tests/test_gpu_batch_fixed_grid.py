"""Models whose grid does not move (movegrid = 0): a model alone against the correctly
rounded oracle, and a batch of them against each model alone, bit for bit, over several
updates of the masses and of the time step, with and without graph replay and with the
models stepped on their own between two calls of the batch."""
import os

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))
MESHES = [(60, 20), (37, 11), (45, 27)]


def _model(nelx, nelz, precision):
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    p["movegrid"] = 0
    return sweep.make_model(p, precision)


def _differing(a, b):
    diff = [f for f in state.State.FIELDS if not np.array_equal(getattr(a, f), getattr(b, f))]
    return diff + [k for k in ("nloop", "time", "dt", "dt_elastic") if getattr(a.clock, k) != getattr(b.clock, k)]


@pytest.mark.gpu
def test_fixed_grid_alone_bitwise_equal_to_oracle():
    from tests import oracle_lib as ol
    print("case: 45x27 elements, fixed grid, 43 steps against the oracle", flush=True)
    gp, st, m = _model(45, 27, abi.PREC_FP64)
    with m:
        m.download()
        ref = st.copy()
        cord = st.cord.copy()
        m.step(43)
        m.download()
    assert ol.step(gp, ref, 43, cr=True) == 0
    assert not [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
    assert np.array_equal(st.cord, cord) and st.vel.any()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [abi.PREC_FP64, abi.PREC_MIXED, abi.PREC_MIXED_STORAGE])
@pytest.mark.parametrize("graph", [False, True])
def test_fixed_grid_batch_equals_models_alone(precision, graph):
    n1, n2, n3 = 33, 4, 36
    print("case: precision %d, fixed grids, batch %d steps (graph %s), alone %d, batch %d" % (precision, n1, graph, n2, n3),
          flush=True)
    alone = []
    for nelx, nelz in MESHES:
        gp, st, m = _model(nelx, nelz, precision)
        with m:
            m.step(n1 + n2 + n3)
            m.download()
        alone.append(st)
    models = [_model(nelx, nelz, precision)[2] for nelx, nelz in MESHES]
    for steps in (n1, n3):
        with sweep.Batch(models) as b:
            b.set_graph(graph)
            b.step(20)
            b.step(steps - 20)
        if steps == n1:
            for m in models:
                m.step(n2)
    diff = []
    for m, ref in zip(models, alone):
        m.download()
        diff.append(_differing(m.state, ref))
        m.close()
    assert diff == [[], [], []]
