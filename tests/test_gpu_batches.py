"""The batch form at the ends of its range of snapshot counts."""
import numpy as np
import pytest

from fastimagingpipe_amd import hip
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


def test_batches_on_two_streams_keep_their_counts(fip):
    """A batch whose turn has not come yet keeps the counts it was called with,
    although another one with other counts is called on another stream."""
    image, nbl, tile, S = 512, 3000, 32, 64
    cell = 1.45e-5 * 1024 / image
    vr, vi, B, V = (a[np.arange(S) % 3] for a in snapshots(29, 3, nbl, image, cell))
    counts = [np.full(S, nbl, np.int32), np.where(np.arange(S) % 3 == 1, nbl // 2, nbl).astype(np.int32)]
    ref = [fip.batch_host(vr, vi, B, V, nv, nbl, image, cell, tile) for nv in counts]
    assert not np.array_equal(ref[0], ref[1])
    dev = [hip.DeviceArray(np.ascontiguousarray(a)) for a in (vr, vi, B, V)]
    out = [hip.DeviceArray(nbytes=ref[0].nbytes) for _ in range(2)]
    other = hip.Stream()
    for which in (0, 0, 1):   # the first two one after the other on the library's stream
        fip.batch_device(dev[0].addr, dev[1].addr, fip.VIS_F32, dev[2].addr, dev[3].addr, counts[which], nbl, S, nbl,
                         image, cell, tile, out[which].addr, stream=other.addr if which else 0)
    hip.synchronize()
    for which in (0, 1):
        got = out[which].to_host(np.float32, ref[0].shape)
        assert np.array_equal(got.view(np.uint32), ref[which].view(np.uint32)), which
