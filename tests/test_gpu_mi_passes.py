"""The histogram passes of the linear stage where their launches differ: a level of few samples, blocks
of samples below and above the count that keeps copies of the histogram, bins whose copies no longer
fit, batches of two to four transforms, a constant background (most samples in one cell), and values
at the top of the range. The cells are integers: a pass of several transforms, and a pass split over
other blocks, give those of the plain pass exactly; the value is the f64 oracle's to 1e-5 (f32
coordinates and weights, the bound of the other sampled-MI tests)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from fastwarp_amd._abi import Affine, LinearTransform, MiBinning
from fastwarp_amd.backend import HipBackend, MiLevel
from tests import cases
from tests.test_gpu_mi import fixed_bins, smooth_vol

pytestmark = pytest.mark.gpu


def level_of(backend, count, bins, background):
    g = cases.grid((40, 36, 30), (1.2, 1.0, 1.4), (-20.0, -15.0, -18.0))
    f = smooth_vol(g, (0, 0, 0))
    m = smooth_vol(g, (1.1, -0.8, 0.6), 0.3)
    if background:
        i, j, k = cases.coords(g)
        out = (i < 14) | (j < 10) | (k > 22)
        f, m = np.where(out, 0.0, f), np.where(out, 0.0, m)
    pts = np.array([g.index_to_point(p) for p in np.random.default_rng(9).uniform([4, 4, 4], np.array(g.shape_xyz) - 5, size=(count, 3))])
    b = MiBinning.from_ranges(bins, (f.min(), f.max()), (m.min(), m.max()))
    fb = fixed_bins(g, f, pts, b)
    centre = tuple(g.index_to_point(np.array(g.shape_xyz) / 2))
    return g, m, pts, fb, b, centre, MiLevel(backend, backend.upload_image(g, m), pts, fb, b)


@pytest.mark.parametrize("count,bins,background", [(1, 32, False), (256, 32, True), (257, 32, True), (5000, 5, False), (70000, 32, True), (40000, 64, True)])
def test_passes_give_the_same_cells(backend, count, bins, background):
    g, m, pts, fb, b, centre, level = level_of(backend, count, bins, background)
    rng = np.random.default_rng(3)
    ts = [LinearTransform.make(0, np.concatenate([rng.normal(0, 0.02, 3), rng.normal(0, 0.5, 3)]), centre) for _ in range(4)]
    want = [level.value(t) for t in ts]
    if count > 1:
        exact = oracle.mi_sampled(b, g, m, pts, fb, ts[0])["value"]
        # five bins leave one bin a side and a value of zero: there only the weights' f32 rounding (6e-8) is left
        assert abs(want[0] - exact) <= 1e-5 * abs(exact) + 1e-7
    cells = level.histogram(ts[0], bins)
    try:
        # blocks of more than 256 samples keep copies of the histogram; those of 300 blocks have fewer
        for blocks in (1, 16, 34, 300):
            backend.set_tuning("mi.max_blocks", blocks)
            for threads in (256, 512, 1024):
                backend.set_tuning("mi.threads", threads)
                j, f, n = level.histogram(ts[0], bins)
                assert n == cells[2] and np.array_equal(j, cells[0]) and np.array_equal(f, cells[1]), (blocks, threads)
                for k in (2, 3, 4):
                    assert list(level.values(ts[:k])) == want[:k], (blocks, threads, k)
    finally:
        backend.set_tuning("mi.max_blocks", -1)
        backend.set_tuning("mi.threads", -1)


def test_values_at_the_top_of_the_range(backend):
    # the identity on the voxel centres: many samples carry the moving maximum itself
    g = cases.grid((32, 32, 32))
    f = cases.image(g, 1)
    m = np.minimum(cases.image(g, 2), 0.6)
    i, j, k = cases.coords(g)
    pts = np.stack([i, j, k], 1)
    b = MiBinning.from_ranges(32, (f.min(), f.max()), (m.min(), m.max()))
    fb = fixed_bins(g, f, pts, b)
    level = MiLevel(backend, backend.upload_image(g, m), pts, fb, b)
    t = LinearTransform.make(0, np.zeros(6))
    joint, marginal, valid = level.histogram(t, 32)
    assert valid == g.n and marginal.sum() == g.n
    assert abs(joint.sum() - g.n) <= 1e-6 * g.n
    want = oracle.mi_sampled(b, g, m, pts, fb, t)["value"]
    assert abs(level.value(t) - want) <= 1e-5 * abs(want)


def test_an_image_beyond_32_bit_byte_offsets_gives_the_cells_of_its_part():
    """An image of 2^30 voxels and more takes the 64-bit form of the gathers. All its content lies near its far
    corner and is that of a small image on the same lattice; points and translations are multiples of 1/8
    around a centre that is their mean, so the f32 coordinates of both are exact and the cells, values and
    derivatives equal."""
    n, at = 48, (940, 960, 970)
    small = cases.grid((n, n, n), (1.0, 1.0, 1.0), tuple(float(q) for q in at))
    big = cases.grid((1024, 1024, 1025), (1.0, 1.0, 1.0), (0.0, 0.0, 0.0))
    assert big.n >= 1 << 30
    m = smooth_vol(small, (0.5, -0.25, 0.75))
    offsets = np.random.default_rng(5).integers(-120, 121, size=(3000, 3)) / 8.0
    pts = np.array(at) + 24.0 + np.concatenate([offsets, -offsets])
    bins = MiBinning.from_ranges(32, (0.0, 1.0), (m.min(), m.max()))
    fb = np.random.default_rng(6).integers(2, 30, size=len(pts)).astype(np.uint32)
    ts = [LinearTransform.make(0, np.array([0.0, 0.0, 0.0, 0.125 * q, -0.25 * q, 0.375]), tuple(np.array(at) + 24.0)) for q in range(4)]
    b = HipBackend(0)
    try:
        src = b.upload_image(small, m)
        results = []
        for image in (src, b.warp_through_field(src, b.zero_field(big))):
            level = MiLevel(b, image, pts, fb, bins)
            results.append(([level.histogram(t, 32) for t in ts], [level.value(t) for t in ts],
                            [list(level.values(ts[:k])) for k in (2, 3, 4)], [level.value_and_derivative(t) for t in ts]))
        (cells, values, batches, gradients), (cells_b, values_b, batches_b, gradients_b) = results
        for (j, f, c), (jb, fb_, cb) in zip(cells, cells_b):
            assert c == cb == len(pts) and np.array_equal(j, jb) and np.array_equal(f, fb_)
        assert values == values_b and batches == batches_b
        for (v, d), (vb, db) in zip(gradients, gradients_b):
            assert v == vb and np.array_equal(d, db)
    finally:
        b.close()
