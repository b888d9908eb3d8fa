"""The pruned transforms at the limit of their band.  A first stage of radix R
whose butterflies prune (12, 16 and 32) takes its inputs 0..nz-1 and R-nz..R-1,
nz = ceil(9 R / 32), so a grid of g rows or columns is pruned as long as the
largest |tap| stays below nz g / R: 9/32 of the grid where the plan begins with
32 (4096^2) and 5/16 where it begins with 16.  Plans that begin with 8 (64^2,
256^2) are never pruned, nor is the row pass of 8192^2.
"""
import numpy as np
import pytest

from tests.inputs import direct_pre_rows, rel_rms, rotation

pytestmark = pytest.mark.gpu

FIRST = {128: 16, 512: 16, 1024: 16, 2048: 16, 4096: 32}


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("image", sorted(FIRST))
def test_largest_tap_at_the_band_limit(fip, oracle, image, axis):
    """Largest |tap| at the limit and one on either side of it, along the rows
    (the column pass's band) or the columns (the row pass's), against the sum
    over the taps at eight rows."""
    n, g = 80, fip.grid_size(image)
    R = FIRST[image]
    cell = 2.0 ** -14 * 64 / image
    V = rotation(0.1, 0.3, 0.2).astype(np.float32)
    for off in (-1, 0, 1):
        top = (9 * R + 31) // 32 * (g // R) + off   # of |tap|; a position p reaches floor(p + 4)
        rng = np.random.default_rng(10 * image + 3 * axis + off)
        p = rng.uniform(-1, 1, (n, 2)) * (top - 5)
        p[:, 1 - axis] = rng.uniform(-0.1, 0.1, n) * g
        p[0, axis], p[1, axis] = top - 3.5, 3.5 - top   # taps up to top and down to -top
        B = (p / (cell * g)).astype(np.float32)
        q = B[:, axis].astype(np.float64) * (cell * g)
        assert np.floor(q + 4).max() == top and np.ceil(q - 4).min() == -top
        vr, vi = rng.standard_normal((2, n)).astype(np.float32)
        vr[:2] = 3.0   # the two that touch the limit weigh most
        pre, _, _ = fip.image(vr, vi, B, V, n, image, 1, cell)
        rows = np.unique(np.concatenate([[0, 1, image // 2 - 1, image // 2, image - 1], rng.integers(0, image, 3)]))
        err = rel_rms(pre[0][rows], direct_pre_rows(oracle, vr, vi, B, V, image, cell, rows))
        print(f"image {image} axis {axis} largest tap {top}: pre rel-rms {err:.2e}", flush=True)
        # The bounds of the image tests: 5e-6 up to 1024^2, twice that above.  A
        # tap lost at the limit would show as about 2e-4.
        assert err < (5e-6 if image <= 1024 else 1e-5)
