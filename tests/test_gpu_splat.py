"""The splat's tile and the trigger's place by image size: on either side of
each rule a call gives the bits of the separate image and trigger."""
import numpy as np
import pytest

from tests.inputs import snapshots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("image,nbl", [(64, 300), (512, 4000), (1024, 8000), (2048, 9000), (4096, 9000)])
def test_pipe_equals_image_then_trigger(fip, image, nbl):
    cell, tile = 1.45e-5 * 1024 / image, 32
    vr, vi, B, V = snapshots(3 + image, 3, nbl, image, cell)
    _, img, mx = fip.image(vr, vi, B, V, nbl, image, 3, cell)
    got = fip.fipipe(vr, vi, B, V, nbl, image, 3, cell, tile)
    ref = fip.trigger(img[0], img[1], img[2], mx, tile)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
