"""Block means summed by the tiles themselves or by their own launch.

Tolerance: N^-1 within 1e-12 of the oracle's direct product, as for every tile
kernel.  The two routes add the same partial sums in the same order, so a block
gives the same bits alone (its tiles sum the mean) and beside others that take
the product over the limit of 512 tiles (a launch of its own does)."""
import numpy as np
import pytest

from midapack_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LAM = 32


def _problem(gpu, blocks, mode):
    m = int(blocks.sum())
    rows = {int(n): W.invtt_block(max(int(n), 2 * LAM), LAM, 1.0, 0.2, 1.5) for n in set(blocks)}
    invtt = np.concatenate([rows[int(n)] for n in blocks])
    pix = np.repeat(3 * (np.arange(m) % 97), 3).astype(np.int32) + np.tile(np.arange(3, dtype=np.int32), m)
    return invtt, gpu.Problem(pix, np.tile([1.0, 0.3, -0.2], m), blocks, LAM, invtt,
                              opts=gpu.options(tile_log2=11, tile_variant=3, offset_mode=mode))


# one chunk of 1024; 64 chunks and one around them; a block that is only mean-subtracted
@pytest.mark.parametrize("blocks", [[700], [1024, 1025, 2047], [65536, 65537, 20, 63000], [400000]])
@pytest.mark.parametrize("mode", ["REFERENCE", "NONE"])
def test_block_means_match_oracle_and_other_route(gpu, blocks, mode):
    first = np.array(blocks, np.int32)
    m = int(first.sum())
    many = np.concatenate([first, np.full(513, 1000, np.int32)])  # 513 tiles more
    x = np.random.default_rng(m).standard_normal(int(many.sum())) + 0.7
    gm = getattr(gpu, "MGPU_OFFSET_" + mode)
    invtt, pb = _problem(gpu, first, gm)
    with pb:
        pb.apply_weights(x[:m])
        alone = pb.apply_weights(x[:m])
    with _problem(gpu, many, gm)[1] as pb:
        pb.apply_weights(x)
        beside = pb.apply_weights(x)
    # chunks of 1024 samples start at the same place in both
    assert np.array_equal(alone, beside[:m])
    with O.ninv_mode(O.NINV_DIRECT), O.offset_mode(getattr(O, "OFFSET_" + mode)):
        ref = O.apply_weights(x[:m], first, LAM, invtt)
    assert np.max(np.abs(alone - ref)) <= 1e-12 * np.max(np.abs(ref))


def test_longest_blocks(gpu):
    """one round of the tiles' loads (524288 samples) and one sample more, where the launch takes over"""
    for n in (524288, 524289):
        blocks = np.array([n], np.int32)
        x = np.random.default_rng(n).standard_normal(n) + 0.7
        invtt, pb = _problem(gpu, blocks, gpu.MGPU_OFFSET_REFERENCE)
        with pb:
            out = pb.apply_weights(x)
        with O.ninv_mode(O.NINV_DIRECT), O.offset_mode(O.OFFSET_REFERENCE):
            ref = O.apply_weights(x, blocks, LAM, invtt)
        assert np.max(np.abs(out - ref)) <= 1e-12 * np.max(np.abs(ref)), n


@pytest.mark.parametrize("gap", [0, 5])
def test_partials_of_many_chunks(gpu, gap):
    """more than 8192 chunks of 1024 samples (four a workgroup): blocks that end inside chunks,
    several in one chunk, a last part chunk and samples past the blocks"""
    blocks = np.array([3_000_001, 64, 100, 70, 2_000_000, 1023, 3_400_000 + 777], np.int32)
    m = int(blocks.sum()) + gap
    rows = {int(n): W.invtt_block(max(int(n), 2 * LAM), LAM, 1.0, 0.2, 1.5) for n in set(blocks)}
    invtt = np.concatenate([rows[int(n)] for n in blocks])
    pix = np.repeat(3 * (np.arange(m) % 97), 3).astype(np.int32) + np.tile(np.arange(3, dtype=np.int32), m)
    x = np.random.default_rng(m).standard_normal(m) + 0.7
    with gpu.Problem(pix, np.tile([1.0, 0.3, -0.2], m), blocks, LAM, invtt,
                     opts=gpu.options(offset_mode=gpu.MGPU_OFFSET_REFERENCE)) as pb:
        out = pb.apply_weights(x)
    with O.ninv_mode(O.NINV_DIRECT), O.offset_mode(O.OFFSET_REFERENCE):
        ref = O.apply_weights(x, blocks, LAM, invtt)
    assert np.max(np.abs(out - ref)) <= 1e-12 * np.max(np.abs(ref))
