"""The CC kernel that computes one plane at a time (small levels, and oblique grids of small radius), and
the kernel that walks its planes, on the same grids: every radius, with and without a mask, on axis-aligned,
permuted and oblique axes, against the f64 oracle and against each other. The axis-aligned bounds are those
of the tile tests (two f32 roundings, held to 1e-6 of the range); on oblique grids the gradient is the
difference of two f32 interpolations, held to 1e-5 as in the other oblique tests."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from fastwarp_amd._abi import Grid
from fastwarp_amd.phantom import make_pair
from fastwarp_amd.register import plan_2mm, register_batch, register_resident
from tests import cases
from tests.test_gpu_cc_tiles import PERMUTED, walks
from tests.test_zz_no_alloc import hip, noalloc_pair

pytestmark = pytest.mark.gpu

GRIDS = {
    "axis": cases.grid((34, 17, 23), (1.0, 2.0, 0.5)),
    "permuted": Grid.make((33, 9, 21), (2.0, 2.0, 2.0), (3.0, -2.0, 1.0), PERMUTED),
    "oblique": cases.grid((34, 17, 23), (1.1, 0.9, 1.3), (-12.5, 7.25, -4.0), oblique=0.35),
}


def pair(backend, g, f, m, radius, valid=None):
    df, dm = backend.upload_image(g, f), backend.upload_image(g, m)
    if valid is None:
        (v0, d0), (v1, d1) = backend.cc_value_derivative_pair(df, dm, radius)
    else:
        (v0, d0), (v1, d1) = backend.cc_value_derivative_pair_masked(df, dm, backend.upload_image(g, valid), radius)
    return (v0, backend.download_field(d0)), (v1, backend.download_field(d1))


def holes(g):
    i, j, k = cases.coords(g)
    return ((i >= 3) & (j < 9) & (k != 7) & ((i + 2 * j + 3 * k) % 11 != 0)).astype(float)


@pytest.mark.parametrize("radius", range(1, 9))
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("axes", list(GRIDS))
def test_both_kernels_match_the_oracle(backend, axes, masked, radius):
    g = GRIDS[axes]
    f, m = cases.image(g, 3), cases.image(g, 4)
    valid = holes(g) if masked else None
    bound = 1e-5 if axes == "oblique" else 1e-6
    want = oracle.cc(g, f, m, radius, mask=valid), oracle.cc(g, m, f, radius, mask=valid)
    got = [pair(backend, g, f, m, radius, valid)]
    # a run of seven planes (shorter and longer than the windows' cycles), and one of all planes
    for planes in (7, 64):
        with walks(backend, planes):
            got.append(pair(backend, g, f, m, radius, valid))
    for both in got:
        for (value, field), w in zip(both, want):
            assert abs(value - w["value"]) <= 1e-6 * abs(w["value"])
            assert cases.rel_err(field, w["derivative"]) <= bound
    if axes == "oblique" and radius < (4 if masked else 7):
        # one kernel: a plane's bits do not depend on the run it is computed in
        for both in got[1:]:
            assert all(np.array_equal(a[1], b[1]) for a, b in zip(both, got[0]))


@pytest.mark.parametrize("radius", [1, 3, 4, 8])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 3e38])
def test_a_value_that_is_not_finite_stays_in_its_windows(backend, radius, bad):
    """A voxel whose window holds a NaN or an infinity counts as degenerate (localCC 1, derivative 0,
    cc.rs:270-300 on the same comparisons); every other voxel keeps its bits. A finite value near the
    f32 limit is no special case: the sums are f64."""
    g = GRIDS["axis"]
    f, m = cases.image(g, 5), cases.image(g, 6)
    at = 20 + 34 * (8 + 17 * 11)
    spoilt = f.copy()
    spoilt[at] = bad
    spoilt = spoilt.astype(np.float32).astype(np.float64)
    i, j, k = cases.coords(g)
    near = (abs(i - 20) <= radius) & (abs(j - 8) <= radius) & (abs(k - 11) <= radius)
    for planes in (None, 64):
        if planes is None:
            clean, got = pair(backend, g, f, m, radius), pair(backend, g, spoilt, m, radius)
        else:
            with walks(backend, planes):
                clean, got = pair(backend, g, f, m, radius), pair(backend, g, spoilt, m, radius)
        for (v, d), (_, d_clean) in zip(got, clean):
            assert np.isfinite(v)
            assert np.array_equal(d[~near], d_clean[~near])
            if not np.isfinite(bad):
                assert np.all(d[near] == 0.0)


@pytest.mark.parametrize("size,radius", [((182, 218, 182), 4), ((182, 218, 90), 7), ((40, 33, 21), 8), ((96, 112, 96), 2)])
@pytest.mark.parametrize("oblique", [0.0, 0.35])
def test_the_pair_without_allocation_takes_the_same_launch(backend, size, radius, oblique):
    # runs of several planes and of one, both kernels: the bits of fw_cc_pair, value included
    g = cases.grid(size, (1.1, 0.9, 1.3), oblique=oblique)
    f, m = cases.image(g, 7), cases.image(g, 8)
    values, d0, d1 = noalloc_pair(hip(), g, f, m, radius)
    (v0, e0), (v1, e1) = pair(backend, g, f, m, radius)
    assert values[0] == v0 and values[1] == v1
    assert np.array_equal(d0, e0) and np.array_equal(d1, e1)


@pytest.mark.parametrize("radius,oblique", [(2, 0.35), (4, 0.35), (7, 0.35), (5, 0.0)])
def test_batched_pairs_give_the_bits_of_single_ones(backend, radius, oblique):
    # subjects against one template through the batched launches of both kernels (levels on both sides of the line)
    pairs = [make_pair((96, 112, 96), 2.0, seed=30 + q) for q in range(3)]
    g = cases.grid((96, 112, 96), (2.0, 2.0, 2.0), tuple(pairs[0].grid.origin), oblique=oblique)
    up = lambda v: [backend.upload_image(g, v)]
    plan = plan_2mm(1)
    plan.set_linear([8, 5], [4, 2], [2.0, 1.0])
    plan.set_syn([4, 3, 2], [4, 2, 1], [2.0, 1.0, 0.0])
    plan.cc_radius = radius
    template, moving = up(pairs[0].fixed[0]), [up(p.moving[0]) for p in pairs]
    batch = register_batch(backend, plan, template, moving)
    for got, mov in zip(batch, moving):
        alone = register_resident(backend, plan, template, mov)
        for name in ("forward", "inverse"):
            assert np.array_equal(backend.download_field(getattr(got, name)), backend.download_field(getattr(alone, name))), name
