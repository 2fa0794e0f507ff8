"""The training gradient at the sizes where its tiles can go wrong (32 samples a wave, up
to 256 workgroups of 8 waves): less than a tile, one sample past a tile, one tile past a
wave of every workgroup, samples of weight 0 in a tile and in a whole tile, sample addresses
that are only 4-byte aligned.  Against the float64 CPU reference.  Bound: the sums run
over at most a few thousand FP32 roundings of 6e-8 that add up like a random walk, so
2e-6 of the gradient's norm leaves a factor of several."""
import numpy as np
import pytest

from tests import mlp_ref


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 31, 33, 257, 8192, 8193, 65536 + 32])
def test_gradient_at_tile_edges(n):
    from geoflac_amd import gpu
    from tests.test_zz_no_alloc import _hip, _to_dev
    H = _hip()
    print("case: gradient over %d samples" % n, flush=True)
    rng = np.random.default_rng(n)
    w = (mlp_ref.init(seed=4) + rng.normal(0, 0.05, mlp_ref.NPARAM)).astype(np.float32)
    x = rng.normal(size=(n, 7)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    weight = np.ones(n)
    if n > 33:
        weight[5::11] = 0.0
        weight[32:64] = 0.0
    smp = np.concatenate([x, np.where(weight > 0, t, np.nan)[:, None]], axis=1).astype(np.float32)
    # the samples one float past the start of an allocation
    buf = _to_dev(H, np.concatenate([np.zeros(1, np.float32), smp.ravel()]).astype(np.float32))
    wd, grad = _to_dev(H, w), _to_dev(H, np.full(mlp_ref.NPARAM + 1, np.nan, dtype=np.float32))
    got = np.empty(mlp_ref.NPARAM + 1, dtype=np.float32)
    try:
        at = type(buf)(buf.value + 4)
        assert gpu.lib().gf_mlp_grad_noalloc(at, n, wd, grad, None) == 0
        assert H.hipDeviceSynchronize() == 0
        assert H.hipMemcpy(got.ctypes.data, grad, got.nbytes, 2) == 0   # device to host
    finally:
        for b in (buf, wd, grad):
            H.hipFree(b)
    g = got.astype(np.float64)
    keep = weight > 0
    w64 = w.astype(np.float64)
    lref, gref = mlp_ref.loss_grad(w64, x[keep].astype(np.float64), t[keep].astype(np.float64))
    gref = gref * keep.sum() / n  # (the mean is over every sample)
    assert abs(g[-1] - lref * keep.sum()) <= 2e-6 * lref * keep.sum()
    assert np.linalg.norm(g[:-1] - gref) <= 2e-6 * np.linalg.norm(gref)
