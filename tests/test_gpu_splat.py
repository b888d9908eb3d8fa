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


@pytest.mark.parametrize("tile", [1, 3, 11, 12, 13, 50, 63, 128])
def test_trigger_by_tile_matches_oracle(fip, oracle, tile):
    """Tiles on either side of each form of the trigger: 16-byte loads, several
    or single turns of 4-byte loads, remainders of a wave's 64 places."""
    rng = np.random.default_rng(tile)
    d = rng.uniform(0.0, 1.0, (3, 256, 256)).astype(np.float32)
    top = d.max((1, 2))
    got = fip.trigger(d[0], d[1], d[2], top, tile)
    ref = oracle.trigger(d[0], d[1], d[2], top, tile)
    # sums of up to tile^2 / 64 terms per lane and six more, in FP32: below
    # 262 * 6e-8 each of three factors at most 1
    assert np.abs(got - np.asarray(ref).reshape(got.shape)).max() < 5e-5
