"""Tile lengths and variants of N^-1 chosen by problem size.

Tolerance: N^-1 within 1e-12 of the exact banded product, as for every other
tile kernel (an FFT of 2^15 points rounds to about log2(N) 1e-16)."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


def _product(gpu, blocks, lam, opts):
    m = int(blocks.sum())
    rng = np.random.default_rng(m + lam)
    rows = {int(n): W.invtt_block(int(n), lam, 1.0, 0.2, 1.5) for n in set(blocks)}
    invtt = np.concatenate([rows[int(n)] for n in blocks])
    pix = np.repeat(3 * (np.arange(m) % 97), 3).astype(np.int32) + np.tile(np.arange(3, dtype=np.int32), m)
    x = rng.standard_normal(m) + 0.5
    with gpu.Problem(pix, np.tile([1.0, 0.3, -0.2], m), blocks, lam, invtt, opts=opts) as pb:
        out = pb.apply_weights(x)
    with O.ninv_mode(O.NINV_DIRECT), O.offset_mode(O.OFFSET_SYMMETRIC):
        ref = O.apply_weights(x, blocks, lam, invtt)
    return _rel(out, ref)


@pytest.mark.parametrize("l2", [11, 13, 14])
def test_tile_variants_match_closed_form(gpu, l2):
    """every FP64 variant of the middle tile lengths, with blocks one sample around whole tiles"""
    N = 1 << l2
    lam = N // 4 + 1
    L = N - 2 * (lam - 1)
    blocks = np.array([2 * lam, L - 1, L, L + 1, 3 * L + 17], np.int32)
    blocks = np.maximum(blocks, 2 * lam).astype(np.int32)
    for v in range(1, len(gpu.tile_variants(gpu.MGPU_FP64, l2)) + 1):
        print(f"N 2^{l2} variant {v}", flush=True)
        err = _product(gpu, blocks, lam, gpu.options(tile_log2=l2, tile_variant=v,
                                                     offset_mode=gpu.MGPU_OFFSET_SYMMETRIC))
        assert err <= 1e-12, (v, err)


@pytest.mark.parametrize("lam,n,nb", [(2, 4099, 1), (33, 70001, 2), (300, 30011, 3), (500, 400009, 2), (1500, 200003, 3),
                                      (3000, 100003, 2), (4097, 40009, 2), (8192, 50021, 1)])
def test_chosen_tile_length_matches_closed_form(gpu, lam, n, nb):
    """the length that the launch-time rule picks, from the shortest tiles to the only one a band fits"""
    print(f"lambda {lam}, {nb} x {n}", flush=True)
    err = _product(gpu, np.full(nb, n, np.int32), lam, gpu.options(offset_mode=gpu.MGPU_OFFSET_SYMMETRIC))
    assert err <= 1e-12, err
