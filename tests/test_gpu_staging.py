"""Host transfers shared by the staging threads: the drop-in's uploads and side
effects at sizes around one worker's share (256 KiB), the 4 MiB from which plain
copies are staged and whole chunks.  Whole-number and copied outputs are exact;
the map of a white-noise solve is a 3 x 3 solve per pixel (1e-12)."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1000, 21845, 21846, 32769, 349525, 349526, 524289, 1050001])
def test_dropin_side_effects_at_staging_edges(gpu, m):
    side = max(8, int((m / 7) ** 0.5))  # about 7 hits a pixel: some pixels are cut
    wl = W.make_workload("staging", 1, m, side, side, 1, m, flag_frac=0.01)
    ref = O.gls_solve(wl.pix, wl.weights, wl.signal, wl.noise, wl.block_sizes, 1, wl.invtt, tol=1e-10, maxiter=5)
    got = gpu.pcg_gls(wl.pix, wl.weights, wl.signal, wl.noise, wl.block_sizes, 1, wl.invtt, tol=1e-10, maxiter=5)
    print(f"m={m}: {got.report['n_cut']} pixels cut", flush=True)
    assert np.array_equal(got.pix_local, ref.pix_local) and np.array_equal(got.lindices, ref.lindices)
    assert np.array_equal(got.weights, ref.weights) and np.array_equal(got.signal, ref.signal)
    assert np.max(np.abs(got.x - ref.x)) <= 1e-12 * np.max(np.abs(ref.x))


@pytest.mark.parametrize("m", [524287, 524288, 1600003])
def test_kept_handle_uploads_at_staging_edges(gpu, m):
    """pcg with host signal and noise of just under 4 MiB, 4 MiB and several chunks a worker"""
    wl = W.make_workload("staging", 1, m, 100, 100, 1, m)
    ref = O.gls_solve(wl.pix, wl.weights, wl.signal, wl.noise, wl.block_sizes, 1, wl.invtt, tol=1e-10, maxiter=5)
    with gpu.Problem(wl.pix, wl.weights, wl.block_sizes, 1, wl.invtt) as pb:
        signal, _, _ = pb.precond_build(wl.signal)
        for _ in range(2):
            x, _, _ = pb.pcg(signal, wl.noise, tol=1e-10, maxiter=5)
            assert np.max(np.abs(x - ref.x)) <= 1e-12 * np.max(np.abs(ref.x))
