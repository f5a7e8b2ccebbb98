"""T^T in one pass over chunks of 2048 samples, at the edges of chunks, pieces
(128 samples) and azimuth bins, against the oracle's sequential sums.

Tolerance: 1e-13 of the largest amplitude, as for the other template cases (at
most 5000 terms, summed in another order)."""
import dataclasses

import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ces_len,nx,kw", [
    (2047, 64, dict()), (2048, 127, dict()), (2049, 128, dict(npoly=1)), (4097, 129, dict(npoly=4, nhwp=2)),
    (300, 300, dict(npoly=0, nhwp=0, n_sss_bins=256)),       # the most bins a chunk sorts its samples into
    (5000, 400, dict(npoly=1, nhwp=1, n_sss_bins=257)),      # azimuth bins summed on their own
    (2500, 2500, dict(npoly=16, nhwp=8, n_sss_bins=3)),      # every class slot, one sweep over two chunks
    (2600, 50, dict(npoly=5, nhwp=3, ground=0, delta_t=0.9)),  # time bins of 9 samples
], ids=lambda v: str(v))
def test_transposed_templates_at_edges(gpu, ces_len, nx, kw):
    wl = W.make_templates_workload("edges", 2, 3, ces_len, nx, 8, 5, **kw)
    if wl.meta["npoly"] == 1:  # with a sweep of one sample (it has no slope) and samples before the first sweep
        wl = W.templates_irregular(wl, cut=ces_len - 7, first=3)
    md = wl.meta
    tm = O.Templates(wl.block_sizes, md["nces"], md["ndet"], wl.invtt, npoly=md["npoly"], ground=md["ground"],
                     n_sss_bins=md["n_sss_bins"], nhwp=md["nhwp"], delta_t=md["delta_t"],
                     sampling_freq=md["sampling_freq"], sweeptstamps=md["sweeptstamps"], az=md["az"],
                     az_min=md["az_min"], az_max=md["az_max"], hwp_angle=md["hwp_angle"])
    d = np.random.default_rng(ces_len).standard_normal(wl.m)
    with gpu.Problem(wl.pix, wl.weights, wl.block_sizes, 1, wl.invtt) as pb:
        pb.set_templates(md)
        got, want = pb.templates_apply(gpu.MGPU_TMPL_TT, d), tm.trtvec(d)
        y = np.repeat(wl.invtt, wl.block_sizes) * d
        filt = pb.templates_apply(gpu.MGPU_TMPL_FILTER, y)
        _, Bi = pb.templates_kernel()
    print(f"T^T error {np.abs(got - want).max() / np.abs(want).max():.1e}", flush=True)
    assert np.abs(got - want).max() <= 1e-13 * np.abs(want).max()
    ref = tm.filter(Bi, y)  # B^+ by representative and factor against the stored pseudo-inverses
    assert np.abs(filt - ref).max() <= 1e-9 * np.abs(ref).max()
