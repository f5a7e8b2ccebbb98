"""The two-level apply on maps past the sizes where its form changes: more than 512
workgroups of 256 pixels (Z^T g summed in a launch between) and more than 256 chunks
of 2048 map entries (longer chunks), with odd pixel counts and few columns.

Tolerance: iterates against the oracle within 1e-10 (1 + k), as for every
two-level iterate."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# kept: 131050 pixels (512 workgroups), 131736 (515) and 175234 (525702 map entries: chunks of 4096)
@pytest.mark.parametrize("zn,nx,ny", [(2, 512, 256), (2, 363, 363), (3, 521, 337)])
def test_twolvl_apply_on_large_maps(gpu, zn, nx, ny):
    wl = W.make_workload("twolvl", 16, 1 << 18, nx, ny, 64, nx)
    k = 1
    with O.ninv_mode(O.NINV_REAL_SPECTRUM):
        r = O.gls_solve(wl.pix, wl.weights, wl.signal, wl.noise, wl.block_sizes, wl.lam, wl.invtt, tol=1e-30,
                        maxiter=50, stop_after=k, precond=1, z_2lvl=zn)
    print(f"case: Zn {zn}, {nx} x {ny} pixels, {r.x.size // 3} kept", flush=True)
    with gpu.Problem(wl.pix, wl.weights, wl.block_sizes, wl.lam, wl.invtt,
                     opts=gpu.options(precond=1, z_2lvl=zn)) as pb:
        sig, _, _ = pb.precond_build(wl.signal)
        x, _, rep = pb.pcg(sig, wl.noise, tol=1e-30, maxiter=50, stop_after=k)
    assert rep.iterations == r.iterations == k
    assert np.max(np.abs(x - r.x)) <= 1e-10 * (1 + k) * np.max(np.abs(r.x))
