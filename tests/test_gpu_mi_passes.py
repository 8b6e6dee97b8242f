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
from fastwarp_amd.backend import MiLevel
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


@pytest.mark.parametrize("count,bins,background", [(1, 32, False), (257, 32, True), (5000, 5, False), (70000, 32, True), (40000, 64, True)])
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
        # 2,048 samples a block and more keep copies of the histogram; one block less than that does not
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
