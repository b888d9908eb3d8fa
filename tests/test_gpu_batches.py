"""The batch form at the ends of its range of snapshot counts."""
import numpy as np
import pytest

from tests.inputs import snapshots

pytestmark = pytest.mark.gpu


def test_batch_of_many_small_snapshots(fip):
    """44000 snapshots of 128^2: more column workgroups than one axis of a launch
    holds threads for.  The snapshots repeat with period four, so each window
    gives the bits of the same window of a short batch."""
    image, nbl, tile, S = 128, 4, 64, 44000
    cell = 1.45e-5 * 1024 / image
    vr, vi, B, V = snapshots(91, 4, nbl, image, cell)
    few = np.arange(10) % 4
    ref = fip.batch_host(vr[few], vi[few], B[few], V[few], None, nbl, image, cell, tile)[:4]
    k = np.arange(S) % 4
    got = fip.batch_host(vr[k], vi[k], B[k], V[k], None, nbl, image, cell, tile)
    assert np.isfinite(ref).all() and len(np.unique(ref)) > 4
    assert np.array_equal(got.view(np.uint32), ref[np.arange(S - 2) % 4].view(np.uint32))
