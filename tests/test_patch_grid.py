"""The patch grid of a merged frame (pkv_patch_grid, the arithmetic of the
update and eviction kernels) against the group ids of mega_merge_accum.cu:
100-184: every token is in one place of its group, and what is read for the
places that a patch lacks lies within the frame, for every frame length and
width, also where the last row is short."""
from __future__ import annotations

import numpy as np
import pytest

from pyramidkv import _abi as A

FIRST = [(128, 52), (110, 52), (70, 34), (963, 37), (8192, 4096), (8191, 7)]


def _grid(fseq, width, patch):
    lib = A.lib()
    n = lib.pkv_patch_grid(fseq, width, patch, None, None)
    read, has = np.full((n, patch * patch), -1, np.int32), np.full((n, patch * patch), 7, np.uint8)
    assert lib.pkv_patch_grid(fseq, width, patch, read.ctypes.data, has.ctypes.data) == n
    return n, read, has


def _check(fseq, width, patch):
    n, read, has = _grid(fseq, width, patch)
    t = np.arange(fseq)
    w = min(width, fseq)
    cols = (w - 1) // patch + 1
    gid = (t // w // patch) * cols + (t % w) // patch
    assert n > gid.max(), (fseq, width, patch)
    where = f"{fseq} tokens in rows of {width}, patch {patch}"
    assert read.min() >= 0 and read.max() < fseq, f"{where}: reads token {read.max()}"
    g, m = np.nonzero(has)
    tok = read[g, m]
    assert np.array_equal(np.sort(tok), t), where
    assert np.array_equal(gid[tok], g), where
    assert all((np.diff(tok[g == k]) > 0).all() for k in np.unique(g)[:8]), f"{where}: not in token order"


@pytest.mark.parametrize("fseq,width", FIRST)
def test_reads_stay_in_the_frame(fseq, width):
    for patch in (1, 2, 3):
        _check(fseq, width, patch)


def test_reads_stay_in_the_frame_for_every_width():
    for fseq in range(1, 97):
        for width in range(1, fseq + 2):
            _check(fseq, width, 2)
    rng = np.random.default_rng(3)
    for _ in range(300):
        fseq = int(2 ** rng.uniform(0, 13))
        _check(fseq, int(rng.integers(1, fseq + 2)), int(rng.integers(1, 3 if fseq < 16 else 5)))


def test_no_grid():
    lib = A.lib()
    assert [lib.pkv_patch_grid(*a, None, None) for a in ((0, 4, 2), (16, 0, 2), (16, 4, 0), (8193, 4, 2))] == [0] * 4


def test_a_patch_larger_than_the_frame_is_not_walked():
    """Its places would number p * p whatever the frame holds: from 1560 ** 0.5
    on, and at sizes whose square does not fit 32 bits."""
    walked = lambda fseq, patch: A.lib().pkv_patch_grid(fseq, 52, patch, None, None) > 0
    assert [p for p in range(1, 2000) if walked(1560, p)] == list(range(1, 40))
    assert not any(walked(1560, p) for p in (46341, 65536, 100000, 2**31 - 1))
    assert all(walked(fseq, 2) for fseq in range(1, 9)) and not walked(4, 3)
