"""White noise (lambda 1): the block weights applied inside P, with blocks that
straddle P's chunks of 1024 samples, samples past the last block, flagged
samples and I weights other than 1; the 3 x 3 blocks of the same samples.

Tolerances: cond, hits and the cut bit-exact; FP64 iterates 1e-12 (at most 4096
terms a pixel), mixed precision 1e-6 (FP32 products, refreshed in FP64)."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [[1, 1000, 1024, 1025, 3000, 7], [8192], [5, 6, 7] * 300], ids=["ragged", "one", "tiny"])
@pytest.mark.parametrize("tail", [0, 1500])
@pytest.mark.parametrize("unit", [True, False])
def test_white_noise_solve(gpu, blocks, tail, unit):
    m = sum(blocks) + tail
    wl = W.make_workload("white", 1, m, 16, 9, 1, 3, flag_frac=0.02)
    rng = np.random.default_rng(4)
    inv = rng.uniform(0.5, 2.0, len(blocks))
    w = wl.weights.copy()
    if not unit:
        w[0::3] = rng.uniform(0.8, 1.2, m)
    bs = np.array(blocks, np.int32)
    ref = O.gls_solve(wl.pix, w, wl.signal, wl.noise, bs, 1, inv, tol=1e-30, maxiter=4)
    got = gpu.pcg_gls(wl.pix, w, wl.signal, wl.noise, bs, 1, inv, tol=1e-30, maxiter=4)
    assert np.array_equal(got.cond, ref.cond) and np.array_equal(got.hits, ref.hits)
    assert np.array_equal(got.pix_local, ref.pix_local) and np.array_equal(got.signal, ref.signal)
    print(f"{len(blocks)} blocks, tail {tail}: {np.max(np.abs(got.x - ref.x)) / np.max(np.abs(ref.x)):.1e}", flush=True)
    assert np.max(np.abs(got.x - ref.x)) <= 1e-12 * np.max(np.abs(ref.x))
    mix = gpu.pcg_gls(wl.pix, w, wl.signal, wl.noise, bs, 1, inv, tol=1e-8, maxiter=50,
                      opts=gpu.options(precision=gpu.MGPU_MIXED))
    assert mix.report["converged"] and np.max(np.abs(mix.x - ref.x)) <= 1e-6 * np.max(np.abs(ref.x))
