"""Several batches or models at once, each in a thread and on a stream of its own, whose thermal
steps all need further passes (columns that couple strongly): none may need the GPU for itself.
Every model against itself alone, bit for bit."""
import os
import threading

import numpy as np
import pytest

from geoflac_amd import abi, inp, state, sweep

HERE = os.path.dirname(os.path.abspath(__file__))


def _model(nelx, nelz, factor):
    p = sweep.variant(inp.read_inp(os.path.join(HERE, "golden", "inputs", "box60x20.inp")), nelx, nelz)
    for ph in p["phases"]:
        ph["conduct"] *= factor
    return sweep.make_model(p, abi.PREC_FP64)


@pytest.mark.gpu
@pytest.mark.parametrize("batches", [1, 6])
def test_concurrent_batches_with_further_passes(batches):
    meshes, n = [(131, 70, 400.0), (60, 20, 1.0), (37, 70, 300.0)], 30
    print("case: %d batches at once of %s (cells, conductivity factor), %d steps" % (batches, meshes, n), flush=True)
    alone = []
    for mesh in meshes:
        gp, st, m = _model(*mesh)
        with m:
            m.step(n)
            m.download()
        alone.append(st)
    made = [[_model(*mesh)[2] for mesh in meshes] for _ in range(batches)]
    handles = [sweep.Batch(models) for models in made]
    failed = []

    def run(b):
        try:
            b.step(n // 2)
            b.step(n - n // 2)
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=run, args=(b,)) for b in handles]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    extra, diff = [], []
    for b, models in zip(handles, made):
        b.close()
        stats = [m.therm_stats() for m in models]
        extra.append(sum(s[1] for s in stats))
        assert not any(s[0] for s in stats)
        for m, ref in zip(models, alone):
            m.download()
            diff += [f for f in state.State.FIELDS if not np.array_equal(getattr(m.state, f), getattr(ref, f))]
            m.close()
    print("  further passes %s" % extra, flush=True)
    assert not failed
    assert not diff
    assert min(extra) >= n  # one in every step


@pytest.mark.gpu
def test_concurrent_models_with_further_passes():
    meshes, n = [(131, 70, 400.0), (400, 200, 15.0), (37, 70, 300.0), (700, 150, 5.0)] * 2, 30
    print("case: models at once, %s (cells, conductivity factor), %d steps" % (meshes, n), flush=True)
    made = [_model(*mesh) for mesh in meshes]
    refs = []
    for mesh in meshes[:4]:
        gp, st, m = _model(*mesh)
        with m:
            m.step(n)
            m.download()
        refs.append(st)
    failed = []

    def run(m):
        try:
            for _ in range(3):
                m.step(n // 3)
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=run, args=(m,)) for _, _, m in made]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    extra, diff = [], []
    for (gp, st, m), ref in zip(made, refs * 2):
        stats = m.therm_stats()
        assert stats[0] == 0
        extra.append(stats[1])
        m.download()
        diff += [f for f in state.State.FIELDS if not np.array_equal(getattr(st, f), getattr(ref, f))]
        m.close()
    print("  further passes %s" % extra, flush=True)
    assert not failed
    assert not diff
    assert min(extra) > 0 and sum(extra) >= 4 * n
