"""The tests by which the compositing kernels leave a list entry out (csrc/splat_staged.cuh): of a tile in the
backward pass (negligible_in_tile), of half a tile in the forward pass (negligible_in_part), and which entries take
their general path (needs_care).  Against brute force over the pixel centres, on the host build of the same code and,
on the GPU, the device build of the first against the host's.

What must hold: an entry that is left out reaches no pixel of the tile with alpha >= 1e-8 (the criterion is a
lower bound of q over the pixels' bounding box, so it may keep entries it could have dropped, never the
reverse); it is worth having: nearly every entry that is far below the threshold at every pixel is found; and the two
passes leave out the same, up to entries that change no pixel.
"""
import numpy as np
import pytest

from tests import _native

THRESHOLD = 1e-8


def _pairs(n, seed, scale_px=(0.5, 40.0)):
    """Random Gaussians with the large benchmark's distributions, each paired with a tile around its
    3-sigma box (a few tiles further out as well, where everything is negligible)."""
    r = np.random.default_rng(seed)
    cx, cy = r.uniform(0, 512, n), r.uniform(0, 512, n)
    sx, sy = (np.exp(r.uniform(np.log(scale_px[0]), np.log(scale_px[1]), n)) for _ in range(2))
    theta = r.uniform(-np.pi, np.pi, n)
    alpha0 = 1 / (1 + np.exp(-r.standard_normal(n)))
    c, s = np.cos(theta), np.sin(theta)
    a = c * c / sx**2 + s * s / sy**2
    b = c * s * (1 / sx**2 - 1 / sy**2)
    cc = s * s / sx**2 + c * c / sy**2
    reach = 3.0 * np.maximum(sx, sy) + 24.0
    tile_x = np.floor((cx + r.uniform(-1, 1, n) * reach) / 16) * 16
    tile_y = np.floor((cy + r.uniform(-1, 1, n) * reach) / 16) * 16
    fields = np.stack([cx, cy, a, b, cc, alpha0], axis=1).astype(np.float32)
    tiles = np.stack([tile_x, tile_y], axis=1).astype(np.float32)
    return fields, tiles


def _largest_alpha(fields, tiles):
    """fp64, every pixel centre of every tile."""
    f = fields.astype(np.float64)
    px = tiles[:, 0, None, None].astype(np.float64) + np.arange(16)[None, None, :] - f[:, 0, None, None]
    py = tiles[:, 1, None, None].astype(np.float64) + np.arange(16)[None, :, None] - f[:, 1, None, None]
    q = f[:, 2, None, None] * px * px + 2 * f[:, 3, None, None] * px * py + f[:, 4, None, None] * py * py
    return f[:, 5] * np.exp(-0.5 * q.min(axis=(1, 2)))


@pytest.mark.parametrize("seed,scale_px", [(1, (0.5, 40.0)), (2, (1.0, 20.0)), (3, (0.3, 3.0))])
def test_nothing_visible_is_left_out_and_most_of_the_invisible_is_found(seed, scale_px):
    fields, tiles = _pairs(40_000, seed, scale_px)
    left_out = _native.negligible_in_tile(fields, tiles)
    largest = _largest_alpha(fields, tiles)
    # never the reverse: what is left out is below the threshold at every pixel (1 % for fp32 against fp64)
    assert left_out.any() and (~left_out).any()
    assert largest[left_out].max() < THRESHOLD * 1.01, largest[left_out].max()
    # worth having: what is far below the threshold everywhere is nearly always recognised (the bounding-box
    # minimum is a little smaller than the minimum over the pixel centres)
    clearly_invisible = largest < THRESHOLD * 1e-3
    assert left_out[clearly_invisible].mean() > 0.98, left_out[clearly_invisible].mean()
    # and the centre inside the tile's box means visible, whatever the shape
    inside = (np.abs(fields[:, 0] - tiles[:, 0] - 7.5) <= 7.5) & (np.abs(fields[:, 1] - tiles[:, 1] - 7.5) <= 7.5)
    assert inside.any() and not left_out[inside & (fields[:, 5] > 1e-6)].any()


def test_odd_records_are_kept():
    fields, tiles = _pairs(64, 4)
    fields[:16, 2] = np.nan  # comparisons with NaN are false: kept, and the projection never bins such a record anyway
    fields[16:32, 5] = 0.0   # alpha0 = 0: nothing to see anywhere
    out = _native.negligible_in_tile(fields, tiles)
    assert not out[:16].any() and out[16:32].all()


def test_fraction_of_the_large_benchmark_scene():
    """The figure behind the kernels' instruction counts: with scales from 0.5 to 40 px about a fifth of the
    (tile, Gaussian) pairs of the 3-sigma boxes cannot be seen from their tile."""
    r = np.random.default_rng(1234)
    G, width, height = 20_000, 2048, 2048
    cx, cy = r.uniform(0, width, G), r.uniform(0, height, G)
    sx, sy = (np.exp(r.uniform(np.log(0.5), np.log(40.0), G)) for _ in range(2))
    theta = r.uniform(-np.pi, np.pi, G)
    alpha0 = 1 / (1 + np.exp(-r.standard_normal(G)))
    c, s = np.cos(theta), np.sin(theta)
    cov_xx, cov_yy = c * c * sx**2 + s * s * sy**2, s * s * sx**2 + c * c * sy**2
    a, b, cc = c * c / sx**2 + s * s / sy**2, c * s * (1 / sx**2 - 1 / sy**2), s * s / sx**2 + c * c / sy**2
    rx, ry = 3 * np.sqrt(cov_xx), 3 * np.sqrt(cov_yy)
    x_lo, x_hi = np.clip(np.floor((cx - rx) / 16), 0, 127).astype(int), np.clip(np.floor((cx + rx) / 16), 0, 127).astype(int)
    y_lo, y_hi = np.clip(np.floor((cy - ry) / 16), 0, 127).astype(int), np.clip(np.floor((cy + ry) / 16), 0, 127).astype(int)
    nx, ny = x_hi - x_lo + 1, y_hi - y_lo + 1
    count = nx * ny
    g = np.repeat(np.arange(G), count)
    k = np.arange(count.sum()) - np.repeat(np.cumsum(count) - count, count)
    tiles = np.stack([(x_lo[g] + k % nx[g]) * 16, (y_lo[g] + k // nx[g]) * 16], axis=1).astype(np.float32)
    fields = np.stack([cx, cy, a, b, cc, alpha0], axis=1).astype(np.float32)[g]
    fraction = _native.negligible_in_tile(fields, tiles).mean()
    assert 0.17 < fraction < 0.27, fraction


def _needles(n, seed, short_px, long_px):
    """Long thin Gaussians, each paired with a tile that its ridge passes through or close by."""
    r = np.random.default_rng(seed)
    sx, sy = np.exp(r.uniform(np.log(short_px / 3), np.log(short_px), n)), np.exp(r.uniform(np.log(long_px / 3), np.log(long_px), n))
    theta = r.uniform(-np.pi, np.pi, n)
    tiles = (np.floor(r.uniform(0, 64, (n, 2))) * 16).astype(np.float32)
    c, s = np.cos(theta), np.sin(theta)
    along = r.uniform(-3, 3, n) * sy
    cx = tiles[:, 0] + r.uniform(-2, 17, n) + along * s
    cy = tiles[:, 1] + r.uniform(-2, 17, n) - along * c
    a, b, cc = c * c / sx**2 + s * s / sy**2, c * s * (1 / sx**2 - 1 / sy**2), s * s / sx**2 + c * c / sy**2
    alpha0 = 1 / (1 + np.exp(-r.standard_normal(n)))
    return np.stack([cx, cy, a, b, cc, alpha0], axis=1).astype(np.float32), tiles


@pytest.mark.parametrize("short_px,long_px", [(20, 40), (0.5, 40), (0.5, 300), (0.3, 1000), (0.5, 10000), (0.3, 3000), (0.1, 1000), (0.02, 200)])
def test_both_passes_leave_out_the_same(short_px, long_px):
    fields, tiles = _needles(200_000, 11, short_px, long_px)
    careful, ill, backward_out, forward_out, largest = _native.compositing_choice(fields, tiles)
    assert careful[ill].all()
    # ill shaped entries: one answer, the tile's, whatever rounding has made of q
    assert (forward_out[ill] == backward_out[ill, None]).all()
    # others: what one pass takes and the other does not has an alpha below 1e-8^(1/1.44) at every pixel of that half
    differ = forward_out != backward_out[:, None]
    assert not differ.any() or largest[differ].max() < 3e-6, largest[differ].max()
    # and the halves are worth having: of what is far below the threshold in a half most is left out of it (ridges of less
    # than a third of a pixel pass between pixel centres, which a minimum over the pixels' box cannot know)
    clearly = (largest < THRESHOLD * 1e-3) & ~ill[:, None]
    if clearly.sum() > 1000 and short_px >= 0.3:
        assert forward_out[clearly].mean() > 0.9, forward_out[clearly].mean()


def test_entries_without_care_at_the_limits():
    """Just inside the limits of needs_care(): alpha stays below the clamp wherever q cancels most, and is exactly 0 at
    the place of a pixel that no Gaussian is to reach, in every row of the tallest image."""
    r = np.random.default_rng(12)
    n = 400_000
    a, c = (np.exp(r.uniform(np.log(1e-9), np.log(1e9), n)) for _ in range(2))
    a[: n // 4], c[: n // 8], c[n // 8 : n // 4] = 1.0001e-9, 0.9999e9, 1.0001e-9
    a[n // 4 : n // 3] = 0.9999e9
    b = np.sqrt(a * c * (1 - 1e-5 * (1 + np.exp(r.uniform(np.log(1e-3), np.log(1e4), n))))) * r.choice([-1.0, 1.0], n)
    pixel = np.stack([np.floor(r.uniform(0, 524272, n)), np.floor(r.uniform(0, 524272, n))], axis=1)
    # centres at all distances, the pixel on the ridge as seen along x: dx = -(b / a) dy, or along y
    reach = np.exp(r.uniform(np.log(1e-2), np.log(4e5), n)) * r.choice([-1.0, 1.0], n)
    steep = r.uniform(size=n) < 0.5
    dx, dy = np.where(steep, -b / a * reach, reach), np.where(steep, reach, -b / c * reach)
    cx, cy = np.clip(pixel[:, 0] - dx, -1e6, 1e6), np.clip(pixel[:, 1] - dy, -5e5, 5e5)
    fields = np.stack([cx, cy, a, b, c, np.full(n, 0.98)], axis=1).astype(np.float32)
    fields[:, 5] = np.minimum(fields[:, 5], np.float32(0.98))
    careful = _native.compositing_choice(fields, np.zeros((n, 2), np.float32))[0]
    assert 0.01 < careful.mean() < 0.5
    fields, pixel = fields[~careful], pixel[~careful].astype(np.float32)
    alpha = _native.composited_alpha(fields, pixel)
    assert (alpha > 0.5).sum() > 1000  # the ridge is met
    assert alpha.max() <= 0.98 * (1 + 1e-6)
    pixel[:, 0] = _native.far_away()
    assert (_native.composited_alpha(fields, pixel) == 0).all()
    pixel[:, 1] = np.where(fields[:, 4] > 0, 524271.0, 0.0)
    assert (_native.composited_alpha(fields, pixel) == 0).all()


@pytest.mark.parametrize("field,value", [
    (5, 0.9801), (5, np.nan), (2, 0.9e-9), (2, 1.1e9), (2, -1.0), (2, np.nan), (4, 0.9e-9), (4, 1.1e9), (4, -1.0), (3, 0.999999), (3, np.nan),
    (0, 1.1e6), (0, -1.1e6), (0, np.inf), (1, 5.1e5), (1, -5.1e5), (1, np.nan),
])
def test_entries_beyond_a_limit_need_care(field, value):
    fields = np.array([[5.0, 6.0, 1.0, 0.2, 1.0, 0.5]] * 2, np.float32)
    fields[1, field] = value
    careful = _native.compositing_choice(fields, np.zeros((2, 2), np.float32))[0]
    assert not careful[0] and careful[1]


@pytest.mark.gpu
def test_device_build_decides_like_the_host_build(gpu):
    fields, tiles = _pairs(100_000, 7)
    host = _native.negligible_in_tile(fields, tiles)
    device = _native.negligible_in_tile(fields, tiles, device=True)
    # the two differ in the last bits of exp2: only entries within a percent of the threshold may fall either way
    largest = _largest_alpha(fields, tiles)
    differ = host != device
    assert differ.mean() < 1e-3
    assert np.all(np.abs(np.log(largest[differ] / THRESHOLD)) < 12.0) if differ.any() else True
    assert largest[device].max() < THRESHOLD * 1.01
