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


@pytest.mark.parametrize("image,S", [(64, 511), (64, 512), (256, 31), (256, 32), (512, 7), (512, 8)])
def test_batch_on_both_sides_of_the_splat_tile_rule(fip, image, S):
    """512 tiles of 64 pixels and one snapshot less: each window gives the bits
    of the same three snapshots imaged one by one and triggered."""
    nbl, tile = 400, 32
    cell = 1.45e-5 * 1024 / image
    vr, vi, B, V = snapshots(17 + image, 3, nbl, image, cell)
    img, mx = zip(*[fip.image(vr[s:s + 1], vi[s:s + 1], B[s:s + 1], V[s:s + 1], nbl, image, 1, cell)[1:] for s in range(3)])
    k = np.arange(S) % 3
    got = fip.batch_host(vr[k], vi[k], B[k], V[k], None, nbl, image, cell, tile)
    for r in range(3):
        q = [(r + j) % 3 for j in range(3)]
        ref = fip.trigger(img[q[0]][0], img[q[1]][0], img[q[2]][0], np.array([mx[j][0] for j in q]), tile)
        assert np.array_equal(got[r::3].view(np.uint32), np.broadcast_to(ref.view(np.uint32), got[r::3].shape))
