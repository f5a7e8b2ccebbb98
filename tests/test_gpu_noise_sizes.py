"""The noise-model builder at block lengths around its chains of 256 x 64 terms
and FFT steps of 16 points, piece by piece against the oracle's functions: the
fitted parameters reach the objective that scipy's fit reaches (to 1e-12 of it:
a sum of n/2 squares rounds to about sqrt(n) 1e-16), and the rows are the
apodised inverse transform of the model at those parameters (to 1e-10: powers
and an FFT of at most 2^17 points)."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import noise as N

pytestmark = pytest.mark.gpu

FS = 10.0


@pytest.mark.parametrize("lens", [[300, 512, 513], [8191, 8192, 8193], [16384, 16385, 16640], [32767, 32768, 33025]], ids=str)
def test_noise_invtt_at_edges(gpu, lens):
    lam = min(200, min(lens) // 4)
    x = np.concatenate([W.one_over_f_noise(np.random.default_rng([5, n]), n, 1.0, 0.2, 1.5) for n in lens])
    _, rpar = N.compute_invtt(x, lens, lam, FS, "chebwin")
    out, par = gpu.noise_invtt(x, np.array(lens, np.int32), lam, FS)
    t = 0
    for b, n in enumerate(lens):
        f, psd = N.periodogram(x[t:t + n], FS)
        t += n
        cost = [np.sum((N.logpsd_model(f[1:], *p) - np.log10(psd[1:])) ** 2) for p in (par[b], rpar[b])]
        model = N.inversepsd_model(np.fft.rfftfreq(n, 1.0 / FS), 10 ** -par[b, 0], *par[b, 1:])
        row = N.apod_window(lam) * np.fft.irfft(model, n=n)[:lam]
        err = np.max(np.abs(out[b * lam:(b + 1) * lam] - row)) / np.max(np.abs(row))
        print(f"n={n}: cost {cost[0]!r} against {cost[1]!r}, row error {err:.1e}", flush=True)
        assert cost[0] <= cost[1] * (1 + 1e-12)
        assert err <= 1e-10
