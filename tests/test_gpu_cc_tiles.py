"""The CC kernels at the edges of their tiles (32 x 8 voxels over a run of planes) and of their windows,
against the f64 oracle: one voxel less and more than a tile, runs shorter and longer than a cycle of the
z pass, grids thinner than the window, permuted and flipped axes, masks, and windows of one value. Every
grid here is small enough for the kernel of one plane; a run set in the tuning table gives it to the
walking kernel. The sums are f64, so the derivative's error is the f32 rounding of
its gradient and of the result (two roundings, 1.2e-7 of a voxel's value, held to 1e-6 of the range)
and the value's the f32 rounding of the block partials (6e-8, held to 1e-6). The spacings are powers of two:
the probes half a spacing away then lie at half a voxel exactly, in the oracle too.

A window of one value v has a variance of zero up to the rounding of the sum of its squares (n v^2 2^-53 a
few times, exactly zero where the squares' sum fits 53 bits). Where both images are flat, the product of
two such residues lies below the epsilon of cc.rs:270-300 while n v^2 < 2^25 (v < 214 at radius 4), and the window
is degenerate as in the oracle. Beyond that, and where one image alone is flat, the classification rests on
rounding errors in the oracle as well, and only the derivative (zero up to the residue) is compared."""
from __future__ import annotations

import contextlib

import numpy as np
import pytest

import oracle
from fastwarp_amd._abi import Grid
from tests import cases

pytestmark = pytest.mark.gpu

PERMUTED = np.array([[0.0, 0.0, -1.0], [1.0, 0.0, 0.0], [0.0, -1.0, 0.0]])


@contextlib.contextmanager
def walks(backend, planes):
    """Runs of `planes` planes in every block of the walking kernel (any number of blocks is enough)."""
    backend.set_tuning("cc.tile_z", planes)
    backend.set_tuning("cc.min_blocks", 1)
    try:
        yield
    finally:
        backend.set_tuning("cc.tile_z", -1)
        backend.set_tuning("cc.min_blocks", -1)


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
    f, m = cases.image(g, 1), cases.image(g, 2)
    compare(backend, g, f, m, radius)
    with walks(backend, 64):
        compare(backend, g, f, m, radius)


@pytest.mark.parametrize("radius", [2, 4])
def test_permuted_axes_and_masks(backend, radius):
    g = Grid.make((34, 10, 21), (2.0, 2.0, 2.0), (3.0, -2.0, 1.0), PERMUTED)
    f, m = cases.image(g, 3), cases.image(g, 4)
    compare(backend, g, f, m, radius)
    i, j, k = cases.coords(g)
    compare(backend, g, f, m, radius, valid=((i >= 3) & (j < 9) & (k != 7)).astype(float))


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("radius", range(1, 9))
@pytest.mark.parametrize("tile_z", [1, 5, 16, 37])
def test_z_runs(backend, tile_z, radius, masked):
    # 37 planes: more than two cycles of the widest window's z pass (17 planes), no multiple of the runs
    g = cases.grid((40, 20, 37))
    f, m = cases.image(g, 5), cases.image(g, 6)
    i, j, k = cases.coords(g)
    with walks(backend, tile_z):
        compare(backend, g, f, m, radius, valid=((i + j + 2 * k) % 7 != 0).astype(float) if masked else None)


@pytest.mark.parametrize("plateau", [1.0, 0.0, 3000.0, 0.6, 0.7, 100.3])
def test_windows_of_one_value_are_degenerate(backend, plateau):
    # half of the volume holds one value, beyond a window of the other half: localCC 1, derivative 0
    g = cases.grid((48, 24, 24))
    i, _, _ = cases.coords(g)
    f = np.where(i < 24, plateau, cases.image(g, 7)).astype(np.float32).astype(np.float64)
    m = np.where(i < 24, 0.77 * plateau if plateau not in (0.0, 1.0, 3000.0) else plateau, cases.image(g, 8))
    m = m.astype(np.float32).astype(np.float64)
    want = oracle.cc(g, f, m, 4)["value"]
    for planes in (None, 64):
        with walks(backend, planes) if planes else contextlib.nullcontext():
            (v0, d0), _ = backend.cc_value_derivative_pair(backend.upload_image(g, f), backend.upload_image(g, m), 4)
        assert abs(v0 - want) <= 1e-6
        assert np.all(backend.download_field(d0)[i < 20] == 0.0)


@pytest.mark.parametrize("plateau", [0.6, 100.3, 3000.3])
def test_one_flat_image_leaves_no_derivative_beyond_its_residue(backend, plateau):
    # the moving image varies everywhere, so its gradient does not hide the coefficient: the residue of s_ff
    # and s_fm is below 1e-12 of the varying windows' moments, and so is the derivative of their range
    g = cases.grid((48, 24, 24))
    i, _, _ = cases.coords(g)
    scale = max(1.0, plateau)
    f = np.where(i < 24, plateau, scale * cases.image(g, 7)).astype(np.float32).astype(np.float64)
    m = (scale * cases.image(g, 8)).astype(np.float32).astype(np.float64)
    want = oracle.cc(g, f, m, 4)["derivative"]
    for planes in (None, 64):
        with walks(backend, planes) if planes else contextlib.nullcontext():
            (_, d0), _ = backend.cc_value_derivative_pair(backend.upload_image(g, f), backend.upload_image(g, m), 4)
        got = backend.download_field(d0)
        assert np.max(np.abs(got[i < 20])) <= 1e-12 * np.max(np.abs(want))
        assert np.max(np.abs(got[i >= 20] - want[i >= 20])) <= 1e-6 * np.max(np.abs(want))
