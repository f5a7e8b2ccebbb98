"""The two-level apply at the edges of its rule: Z^T g summed by the apply's own
workgroups (at most 16 columns) or in a launch between, one column, maps of one
chunk and of several, odd sizes.

Tolerance: iterates against the oracle within 1e-10 (1 + k), as for every
two-level iterate."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zn,nx,ny", [(1, 5, 7), (3, 33, 31), (16, 37, 41), (17, 37, 41), (5, 64, 61)])
def test_twolvl_apply_sizes(gpu, zn, nx, ny):
    wl = W.config_small(seed=zn + nx, ndet=4, nsamp=8192, nx=nx, ny=ny, lam=64)
    print(f"case: Zn {zn}, {nx} x {ny} pixels", flush=True)
    k = 2
    with O.ninv_mode(O.NINV_REAL_SPECTRUM):
        r = O.gls_solve(wl.pix, wl.weights, wl.signal, wl.noise, wl.block_sizes, wl.lam, wl.invtt, tol=1e-30,
                        maxiter=50, stop_after=k, precond=1, z_2lvl=zn)
    with gpu.Problem(wl.pix, wl.weights, wl.block_sizes, wl.lam, wl.invtt,
                     opts=gpu.options(precond=1, z_2lvl=zn)) as pb:
        sig, _, _ = pb.precond_build(wl.signal)
        x, _, rep = pb.pcg(sig, wl.noise, tol=1e-30, maxiter=50, stop_after=k)
    assert rep.iterations == r.iterations == k
    assert np.max(np.abs(x - r.x)) <= 1e-10 * (1 + k) * np.max(np.abs(r.x))
