"""fip_image's read-back: the ring of pinned chunks (more chunks than slots, a
last partial chunk, fewer threads than its most) and the plain copy below it
give the bits of one snapshot at a time."""
import numpy as np
import pytest

from tests.inputs import snapshots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("image,nsnap", [(128, 2), (128, 41), (128, 130), (512, 3), (1024, 3), (2048, 5)])
def test_image_readback_equals_single_snapshots(fip, image, nsnap):
    cell, nbl = 1.45e-5 * 1024 / image, 1500
    vr, vi, B, V = snapshots(50 + image, nsnap, nbl, image, cell)
    pre, img, mx = fip.image(vr, vi, B, V, nbl, image, nsnap, cell)
    for s in range(nsnap):
        q = slice(s, s + 1)
        p1, i1, m1 = fip.image(np.asarray(vr)[q], np.asarray(vi)[q], np.asarray(B)[q], np.asarray(V)[q], nbl, image, 1,
                               cell)
        assert np.array_equal(pre[s].view(np.uint32), p1[0].view(np.uint32)), s
        assert np.array_equal(img[s].view(np.uint32), i1[0].view(np.uint32)), s
        assert mx[s] == m1[0] == img[s].max()
