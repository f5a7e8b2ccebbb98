"""P^T at every remainder of its steps: pixels with 1 to 35 hits, mixed with
pixels of fewer hits (padding), with and without I weights.

No tolerance: a pixel's sums run over its hits in time order, so NumPy's
sequential sums of the same terms give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit", [True, False])
def test_pt_widths(gpu, unit):
    rng = np.random.default_rng(5)
    for width in list(range(1, 36)) + [47, 48, 49, 64]:
        npix = 64 + 5
        hits = np.where(np.arange(npix) % 3 == 1, max(1, width - width // 2), width)
        order = rng.permutation(np.repeat(np.arange(npix), hits))
        m = order.size
        w = rng.standard_normal((m, 3))
        if unit:
            w[:, 0] = 1.0
        pix = (3 * order[:, None] + np.arange(3)).astype(np.int32).ravel()
        y = rng.standard_normal(m)
        with gpu.Problem(pix, w.ravel(), np.array([m], np.int32), 1, np.ones(1)) as pb:
            out = pb.trmatvec(y)
        ref = np.zeros((npix, 3))
        for t in range(m):
            ref[order[t]] += w[t] * y[t]
        assert np.array_equal(out, ref.ravel()), width
