"""Edits of a reference-layout world whose block pool holds more than 2^32
words (16 GiB): a chunk that names a block past the 2^23rd is written there,
and the first block, whose words have the same number modulo 2^32, keeps its
own."""
import numpy as np
import pytest

import vt

pytestmark = pytest.mark.gpu


def test_edits_past_two_to_the_32_words(ctx):
    n, high = 16, 2 ** 23
    chunks = np.zeros(8, np.uint32)
    chunks[:3] = 1, high + 1, high + 2   # 512 words each
    pool = np.zeros((high + 2) * 512, np.uint32)
    atlas = np.full(256 ** 3, 0xFF202020, np.uint32)
    w = vt.World.brickmap(ctx, n, chunks, pool, atlas)
    rng = np.random.default_rng(2)
    # x < 8, y < 8: the first chunk; x >= 8: the second; y >= 8: the third
    base = rng.permutation(512)[:100]
    at = np.stack([base % 8, base // 8 % 8, base // 64], 1)
    xyz = np.vstack([at, at + (8, 0, 0), at + (0, 8, 0)]).astype(np.uint32)
    for shift in (0, 1000):
        val = (1 + shift + np.arange(len(xyz))).astype(np.uint32)
        w.set_voxels(xyz, val)
        assert np.array_equal(w.get_voxels(xyz), val)
    everything = np.stack([v.ravel() for v in np.mgrid[0:n, 0:n, 0:n]], 1).astype(np.uint32)
    assert np.count_nonzero(w.get_voxels(everything)) == len(xyz)
    w.close()
