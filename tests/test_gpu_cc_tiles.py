"""The CC kernel at the edges of its tiles (32 x 8 voxels over a run of planes) and of its windows,
against the f64 oracle: one voxel less and more than a tile, runs shorter and longer than a cycle of the
z pass, grids thinner than the window, permuted and flipped axes, masks, and windows of one value,
whose variance is exactly zero. The sums are f64, so the derivative's error is the f32 rounding of
its gradient and of the result (two roundings, 1.2e-7 of a voxel's value, held to 1e-6 of the range)
and the value's the f32 rounding of the block partials (6e-8, held to 1e-6). The spacings are powers of two:
the probes half a spacing away then lie at half a voxel exactly, in the oracle too."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from fastwarp_amd._abi import Grid
from tests import cases

pytestmark = pytest.mark.gpu

PERMUTED = np.array([[0.0, 0.0, -1.0], [1.0, 0.0, 0.0], [0.0, -1.0, 0.0]])


def compare(backend, g, f, m, radius, valid=None, bound=1e-6):
    df, dm = backend.upload_image(g, f), backend.upload_image(g, m)
    if valid is None:
        (v0, d0), (v1, d1) = backend.cc_value_derivative_pair(df, dm, radius)
    else:
        (v0, d0), (v1, d1) = backend.cc_value_derivative_pair_masked(df, dm, backend.upload_image(g, valid), radius)
    for v, d, want in ((v0, d0, oracle.cc(g, f, m, radius, mask=valid)), (v1, d1, oracle.cc(g, m, f, radius, mask=valid))):
        assert abs(v - want["value"]) <= 1e-6 * abs(want["value"])
        assert cases.rel_err(backend.download_field(d), want["derivative"]) <= bound


@pytest.mark.parametrize("radius", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("size", [(31, 7, 9), (32, 8, 10), (33, 9, 23), (65, 17, 4), (5, 3, 40)])
def test_tile_edges(backend, size, radius):
    g = cases.grid(size, (1.0, 2.0, 0.5))
    compare(backend, g, cases.image(g, 1), cases.image(g, 2), radius)


@pytest.mark.parametrize("radius", [2, 4])
def test_permuted_axes_and_masks(backend, radius):
    g = Grid.make((34, 10, 21), (2.0, 2.0, 2.0), (3.0, -2.0, 1.0), PERMUTED)
    f, m = cases.image(g, 3), cases.image(g, 4)
    compare(backend, g, f, m, radius)
    i, j, k = cases.coords(g)
    compare(backend, g, f, m, radius, valid=((i >= 3) & (j < 9) & (k != 7)).astype(float))


@pytest.mark.parametrize("tile_z", [1, 5, 64])
def test_z_runs(backend, tile_z):
    g = cases.grid((40, 20, 37))
    f, m = cases.image(g, 5), cases.image(g, 6)
    backend.set_tuning("cc.tile_z", tile_z)
    try:
        compare(backend, g, f, m, 4)
    finally:
        backend.set_tuning("cc.tile_z", -1)


@pytest.mark.parametrize("plateau", [1.0, 0.0, 3000.0])
def test_windows_of_one_value_are_degenerate(backend, plateau):
    # half of the volume holds one value, beyond a window of the other half: localCC 1, derivative 0
    g = cases.grid((48, 24, 24))
    i, _, _ = cases.coords(g)
    f = np.where(i < 24, plateau, cases.image(g, 7))
    m = np.where(i < 24, plateau, cases.image(g, 8))
    (v0, d0), _ = backend.cc_value_derivative_pair(backend.upload_image(g, f), backend.upload_image(g, m), 4)
    assert abs(v0 - oracle.cc(g, f, m, 4)["value"]) <= 1e-6
    assert np.all(backend.download_field(d0)[i < 20] == 0.0)
