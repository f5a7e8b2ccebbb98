"""Several tile classes in one launch: items of a batch with different bands and
tile lengths, more classes than one launch takes, and classes that are left out
(longer tiles).

No tolerance: every item must reproduce its solo solve, one class a launch, bit
for bit."""
import numpy as np
import pytest

from midapack_amd import workloads as W

pytestmark = pytest.mark.gpu


# bands whose chosen or forced tiles are 2^10 .. 2^13 samples, the last also 2^14
@pytest.mark.parametrize("lams,log2,precision", [
    ((2, 300), 0, "fp64"),
    ((16, 100, 300, 700, 1200), 0, "fp64"),
    ((16, 100, 300, 700, 1200), 0, "mixed"),
    (tuple(20 + 9 * k for k in range(18)), 10, "fp64"),
    ((40, 64, 1000), 13, "fp64"),
    ((32, 64, 3000), 14, "fp64"),
])
def test_classes_together_match_solo_bitwise(gpu, lams, log2, precision):
    print(f"case: bands {lams}, tile 2^{log2}, {precision}", flush=True)
    prec = gpu.MGPU_FP64 if precision == "fp64" else gpu.MGPU_MIXED
    opts = gpu.options(precision=prec, offset_mode=gpu.MGPU_OFFSET_SYMMETRIC, tile_log2=log2)
    wls = [W.make_workload(f"c{k}", 1 + k % 2, 2 * lam + 3001 + 64 * k, 24, 24, lam, 50 + k)
           for k, lam in enumerate(lams)]
    items = [dict(pix=w.pix, weights=w.weights, signal=w.signal, noise=w.noise, block_sizes=w.block_sizes, lam=w.lam,
                  invtt=w.invtt) for w in wls]
    res = gpu.pcg_batch(items, 24 * 24, tol=1e-30, maxiter=6, opts=opts)
    for w, r in zip(wls, res):
        g = gpu.pcg_gls(w.pix, w.weights, w.signal, w.noise, w.block_sizes, w.lam, w.invtt, tol=1e-30, maxiter=6,
                        opts=opts)
        assert r.report["iterations"] == g.report["iterations"]
        assert np.array_equal(r.x, g.x), w.name
