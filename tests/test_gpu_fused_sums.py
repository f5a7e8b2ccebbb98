"""The map kernels that sum the dots' partials themselves (segments of at most
1024 workgroups, 262144 pixels) against the reduction kernels: the same bits."""
import numpy as np
import pytest

from midapack_amd import workloads as W

pytestmark = pytest.mark.gpu


def _item(wl):
    return dict(pix=wl.pix, weights=wl.weights, signal=wl.signal, noise=wl.noise, block_sizes=wl.block_sizes,
                lam=wl.lam, invtt=wl.invtt)


def _every_pixel_kept(name, nx, ny, seed):
    """12 detectors pass once over every pixel at 12 even angles: no pixel is cut"""
    wl = W.make_workload(name, 12, nx * ny, nx, ny, 16, seed)
    psi2 = np.repeat(2 * np.pi * np.arange(12) / 12, nx * ny)
    wl.weights[1::3], wl.weights[2::3] = np.cos(psi2), np.sin(psi2)
    return wl


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("graph", [0, 1])
def test_small_segment_alone_and_beside_a_large_one(mixed, graph):
    """Alone, a small map and one of exactly 1024 workgroups take the fused
    kernels; in a batch with a map of 1025 workgroups every segment takes the
    reduction kernels.  Maps, residuals and iteration counts stay bit-identical."""
    from midapack_amd import lib as G
    G.init(0)
    small = W.make_workload("small", 2, 30000, 40, 25, 64, 11, fknee_range=(0.05, 0.5))
    edge = _every_pixel_kept("1024 workgroups", 512, 512, 12)
    large = _every_pixel_kept("1025 workgroups", 656, 400, 13)
    grid = 656 * 400
    opts = G.options(precision=G.MGPU_MIXED if mixed else G.MGPU_FP64, offset_mode=G.MGPU_OFFSET_SYMMETRIC, graph=graph)
    items = [_item(w) for w in (small, edge, large)]
    both = G.pcg_batch(items, grid, tol=1e-10, maxiter=25, opts=opts)
    assert len(both[1].pixels) == 1024 * 256 and len(both[2].pixels) == 1025 * 256
    for i, it in enumerate(items[:2]):
        alone = G.pcg_batch([it], grid, tol=1e-10, maxiter=25, opts=opts)[0]
        print(f"item {i}: {alone.report['iterations']} iterations alone, {both[i].report['iterations']} in the batch",
              flush=True)
        assert alone.report["iterations"] == both[i].report["iterations"]
        assert alone.report["res"] == both[i].report["res"]
        assert np.array_equal(alone.x, both[i].x)
