"""Training kernels of the surrogate at the edges of their tiles (16 atoms a tile, 512 partial
rows), against the numpy oracle and against sums in the kernel's own order."""
import os
import sys

import numpy as np
import pytest

from conftest import REPO, surrogate_module

sys.path.insert(0, os.path.join(REPO, "oracle"))
import surrogate as so  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 511, 16 * 512 + 5])
def test_weight_gradient_at_tile_edges(n):
    """FP32 sums of n terms per parameter, each to a few ulp (2^-24): 1e-5 of the block's norm
    covers sqrt(n) growth at the largest n with a wide margin."""
    es = surrogate_module()
    rng = np.random.default_rng(n)
    p = so.Params(seed=3, d_mean=np.zeros(so.ND), d_std=rng.uniform(0.5, 2.0, so.ND), e0=-3.5,
                  s_e=0.5)
    for b in ("b1", "b2", "b3"):
        setattr(p, b, 0.1 * rng.normal(size=getattr(p, b).shape))
    p.set_flat(p.flat().astype(np.float32).astype(np.float64))
    p.d_std = p.d_std.astype(np.float32).astype(np.float64)
    model = es.Model(p.flat(), p.d_mean, p.d_std, p.e0, p.s_e)
    model.upload()
    dn, U, cE = (rng.normal(size=s).astype(np.float32) for s in ((n, 32), (n, 32), n))
    d = [es.Dev.of(a) for a in (dn, U, cE)]
    g0 = rng.normal(size=so.NPARAM).astype(np.float32)  # the entry point adds to grad
    grad = es.Dev.of(g0)
    assert es.lib().surWeightGradGFX950(n, *(a.ptr for a in d), grad.ptr) == 0
    got = grad.get().astype(np.float64) - g0
    _, cache = so.mlp_forward(p, dn.astype(np.float64) * p.d_std + p.d_mean)
    want = so.weight_gradients(p, cache, cE.astype(np.float64), U.astype(np.float64))
    off = 0
    for name in so.Params.NAMES:
        w = getattr(want, name).reshape(-1)
        r = np.linalg.norm(got[off:off + w.size] - w) / (np.linalg.norm(w) + np.sqrt(w.size))
        print(n, name, "%.2e" % r, flush=True)
        assert r < 1e-5, name
        off += w.size
