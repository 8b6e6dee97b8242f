"""Image and field downloads run in pieces of 2^25 values through a bounded pinned buffer: whole volumes
of one value and of three planes, at sizes that end before, on and after a piece's end, come back as the
f32 values that were sent, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from tests import cases

pytestmark = pytest.mark.gpu

PIECE = 1 << 25


@pytest.mark.parametrize("size", [(1, 1, 1), (31, 601, 1801), (512, 256, 256), (33, 251, 4051)])
def test_images_come_back_whole(backend, size):
    g = cases.grid(size)
    v = np.random.default_rng(g.n).standard_normal(g.n).astype(np.float32).astype(np.float64)
    assert np.array_equal(backend.download_image(backend.upload_image(g, v)), v)


@pytest.mark.parametrize("size,over", [((641, 17449, 1), -1), ((210, 221, 241), 0), ((11, 251, 4051), 1), ((22, 251, 4051), PIECE // 3 + 2)])
def test_fields_come_back_whole(backend, size, over):
    g = cases.grid(size)
    assert g.n == PIECE // 3 + over
    v = np.random.default_rng(g.n).standard_normal((g.n, 3)).astype(np.float32).astype(np.float64)
    assert np.array_equal(backend.download_field(backend.upload_field(g, v)), v)
