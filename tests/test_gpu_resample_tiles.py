"""Resampling over the forms its launch tells apart (tiles of 64 x 1 x 1,
16 x 1 x 4 and 16 x 4 x 1 voxels, views one voxel wide, views of 4 GiB) at sizes
that are no multiple of a tile, bit for bit against the oracle."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import transform as T

pytestmark = pytest.mark.gpu
BLEND = T.Blending()


def _map(axis, deg, raw):
    a, c = math.radians(deg), np.asarray(raw) / 2
    i, j = [(1, 2), (2, 0), (0, 1)][axis]
    m = np.eye(3)
    m[i, i] = m[j, j] = math.cos(a)
    m[i, j], m[j, i] = -math.sin(a), math.sin(a)
    return np.hstack([m, (c - m @ c)[:, None]])


@pytest.mark.parametrize("raw,axis,deg,size", [
    ((70, 33, 41), 0, 35.0, (131, 37, 45)),  # turned about x: rows
    ((70, 33, 41), 1, 60.0, (67, 33, 71)),   # about y: 16 x 4 in x and z
    ((70, 33, 41), 1, -86.0, (67, 33, 71)),  # nearly a right angle: rows
    ((41, 70, 33), 2, 50.0, (83, 81, 6)),    # about z: 16 x 4 in x and y
    ((41, 33, 70), 1, 45.0, (15, 3, 3)),     # one partial tile
    ((1, 33, 41), 1, 45.0, (40, 33, 40)),    # one voxel wide: no pairs
    ((2, 33, 1), 1, 30.0, (9, 33, 5)),
])
def test_tiles(raw, axis, deg, size):
    img = np.random.default_rng(sum(raw)).uniform(0.0, 500.0, raw[::-1]).astype(np.float32)
    inv = T.inverse_affine(_map(axis, deg, raw))
    print("tile", raw, axis, deg, size, flush=True)
    got, gw = T.transform_view(img, inv, (-2, -1, -3), size, BLEND)
    ref, rw = O.transform_view(img, inv, (-2, -1, -3), size, BLEND.border, BLEND.range)
    np.testing.assert_array_equal(got, ref)
    np.testing.assert_array_equal(gw, rw)


def test_far_face():
    """Positions on the last voxels, where the upper corner is the mirrored one."""
    raw = np.random.default_rng(1).uniform(0.0, 500.0, (5, 6, 7)).astype(np.float32)
    inv = np.hstack([np.eye(3), [[0.25], [0.5], [0.75]]])
    got, _ = T.transform_view(raw, inv, (0, 0, 0), (9, 8, 7), None)
    ref, _ = O.transform_view(raw, inv, (0, 0, 0), (9, 8, 7), None, None)
    np.testing.assert_array_equal(got, ref)


def test_view_of_four_gigabytes():
    """64-bit addresses: the last planes of a large view, at positions exact in
    float, equal the same planes as a view of their own."""
    import torch
    big = torch.zeros((1025, 1024, 1024), device="cuda")
    big[-4:] = torch.rand((4, 1024, 1024), device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    out, ref = (torch.empty((3, 70, 1030), device="cuda") for _ in range(2))
    print("view of 4 GiB", flush=True)
    for z, raw, o in ((1021.5, big, out), (0.5, big[-4:].contiguous(), ref)):
        T.transform_view_device(raw, np.hstack([np.eye(3), [[0.25], [0.5], [z]]]), (0, 960, 0), (1030, 70, 3), o)
    assert torch.equal(out, ref)
