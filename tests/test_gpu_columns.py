"""The column kernel at the edges of its cases: the gridded band on either side
of the pruned transform's limit, taps clipped at the grid's edge, integer
positions, mirrored records, and (for its exactness) columns of more records
than its threads hold.
"""
import numpy as np
import pytest

from tests.inputs import direct_pre_rows, rel_rms, rotation

pytestmark = pytest.mark.gpu


def positions(kind, g, rng):
    """Grid positions [n, 2] (row, column)."""
    m = g // 2
    if kind.startswith("band"):   # rows up to just inside / outside 9/32 of the grid
        limit = (9 * g) // 32 + (-4 if kind == "band_in" else 3)
        p = rng.uniform(-0.4, 0.4, (500, 2)) * g
        p[:, 0] = np.clip(p[:, 0], 5 - limit, limit - 5)
        p[:2, 0] = limit - 4.5, 4.5 - limit
        return p
    if kind == "edge":   # taps clipped, wrapped by the mirror, or wholly outside
        e = np.array([-m - 5, -m - 3.7, -m - 0.2, -m, -m + 0.3, -m + 3, -m + 3.9, m - 4.1, m - 3, m - 0.5, m, m + 3.2])
        p = np.stack(np.meshgrid(e, np.concatenate([e, rng.uniform(-m, m, 8)])), -1).reshape(-1, 2)
        return np.concatenate([p, p[:, ::-1]])
    if kind == "integer":   # nine taps per axis
        return 3.0 * rng.integers(-m // 3, m // 3 + 1, (500, 2))
    raise ValueError(kind)


@pytest.mark.parametrize("image", [64, 128, 256, 512, 1024])
@pytest.mark.parametrize("kind", ["band_in", "band_out", "edge", "integer"])
def test_columns_match_oracle(fip, oracle, image, kind):
    rng = np.random.default_rng(image + sum(map(ord, kind)))
    g = fip.grid_size(image)
    cell = 2.0 ** -14 * 64 / image   # cell * g = 3 * 2^-9: multiples of 3 are exact positions
    p = positions(kind, g, rng)
    n = p.shape[0]
    B = (p / (cell * g)).astype(np.float32)
    vr, vi = rng.standard_normal((2, n)).astype(np.float32)
    V = rotation(0.1, 0.3, 0.2).astype(np.float32)
    pre, _, _ = fip.image(vr, vi, B, V, n, image, 1, cell)
    ref, _, _ = oracle.image(vr, vi, B, V, image, cell, want_pre=True)
    err = rel_rms(pre[0], ref)
    print(f"{kind} {image}: pre rel-rms {err:.2e}")
    # The bound of the image test at these sizes, whose inputs have the same
    # spread of magnitudes (5e-6, its measured 8.6e-7 times five).
    assert err < 5e-6


@pytest.mark.parametrize("image,n", [(64, 9000), (256, 9000), (1024, 9000), (2048, 9000)])
def test_crowded_columns_do_not_depend_on_the_order(fip, image, n):
    """Records near one axis, several passes of a column's threads: the sums
    are integers, so any order of the visibilities gives the same bits."""
    rng = np.random.default_rng(image)
    g = fip.grid_size(image)
    cell = 2.0 ** -14 * 64 / image
    p = np.stack([rng.uniform(-0.45, 0.45, n) * g, rng.uniform(-6, 6, n)], -1)
    p[::2, 0] = rng.normal(0, 3, n // 2)
    B = (p / (cell * g)).astype(np.float32)
    vr, vi = rng.standard_normal((2, n)).astype(np.float32)
    V = rotation(0.1, 0.3, 0.2).astype(np.float32)
    k = rng.permutation(n)
    a = fip.image(vr, vi, B, V, n, image, 1, cell)[0]
    b = fip.image(vr[k], vi[k], B[k], V, n, image, 1, cell)[0]
    assert np.isfinite(a).all()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 65537, 81920, 81921, 131073, 262145, 524289])
def test_front_end_keeps_every_visibility(fip, oracle, n):
    """Counts around a sorting workgroup's 2048 visibilities and around each
    change of its visibilities per thread.  A visibility lost or taken twice by
    its place would be another one after a permutation: the bits stay the same.
    """
    image, cell = 64, 2.0 ** -14
    rng = np.random.default_rng(n)
    g = fip.grid_size(image)
    p = rng.uniform(-0.5, 0.5, (n, 2)) * g
    B = (p / (cell * g)).astype(np.float32)
    vr, vi = rng.standard_normal((2, n)).astype(np.float32)
    V = rotation(0.1, 0.3, 0.2).astype(np.float32)
    k = rng.permutation(n)
    a = fip.image(vr, vi, B, V, n, image, 1, cell)[0]
    b = fip.image(vr[k], vi[k], B[k], V, n, image, 1, cell)[0]
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    ref = oracle.image(vr, vi, B, V, image, cell, want_pre=True)[0]
    err = rel_rms(a[0], ref)
    print(f"{n}: pre rel-rms {err:.2e}")
    # The int32 quantum: at 524289 a block of 16 rows of one column sums up to
    # 5e3 in magnitude, so one unit is 2e-5, and the 8e3 contributions of a
    # cell (rms value 20) round to 5e-4 together, 2.5e-5 of it; the grid
    # correction amplifies that by at most 40 at the image's edge.
    assert err < 1e-3


@pytest.mark.parametrize("cmax", [0.0, 3067.6, 3068.6, 3069.6, 4700.2, 6139.9, 6143.5])
def test_row_pass_of_the_largest_image(fip, oracle, cmax):
    """8192^2: two rows in two transforms of half the grid.  Columns up to each
    side of g/4 (where the two halves of the band begin to overlap), to g/2 and
    clipped there, against the sum over the taps at sixteen rows."""
    image, n = 8192, 60
    rng = np.random.default_rng(int(10 * cmax))
    g = fip.grid_size(image)
    cell = 2.0 ** -14 * 64 / image
    p = np.stack([rng.uniform(-0.45, 0.45, n) * g, rng.uniform(-1, 1, n) * cmax], -1)
    p[:2, 1] = cmax, -cmax
    p[2:4] = 0.0
    B = (p / (cell * g)).astype(np.float32)
    vr, vi = rng.standard_normal((2, n)).astype(np.float32)
    V = rotation(0.1, 0.3, 0.2).astype(np.float32)
    pre, _, _ = fip.image(vr, vi, B, V, n, image, 1, cell)
    rows = np.unique(np.concatenate([[0, 1, 2, 3, 4095, 4096, 8190, 8191], rng.integers(0, image, 8)]))
    ref = direct_pre_rows(oracle, vr, vi, B, V, image, cell, rows)
    err = rel_rms(pre[0][rows], ref)
    print(f"cmax {cmax}: pre rel-rms {err:.2e}")
    # Twice the bound of the sizes up to 1024 above: a longer transform and the
    # sum that splits it.
    assert err < 1e-5
