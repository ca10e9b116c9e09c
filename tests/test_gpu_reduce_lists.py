"""The voxel reduce at the edges of its split of a brick's boxes over
wavefronts: every workgroup's box overlaps the same bricks, and the number of
workgroups runs over one round's boxes (16), every wavefront's first round (32
and 64) and one more or less, alone and in a batch.  Strands and voxel ints
bitwise against ref32."""
import numpy as np
import pytest

import hairsim
import oracle
from hairsim import scenes
from helpers import assert_bitwise

pytestmark = pytest.mark.gpu

BOXES = (1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 129)


def _groom(boxes, seed):
    """boxes * 128 strands of 2 points (one segment, one box per workgroup of 128) around one place."""
    rng = np.random.default_rng(seed)
    S = boxes * 128 - (boxes > 1) * 5
    aos = np.zeros((S, 3, 2, 4), np.float32)
    aos[:, 0, :, 3] = 1
    aos[:, 0, 0, :3] = rng.uniform(-0.02, 0.02, (S, 3))
    aos[:, 0, 1, :3] = aos[:, 0, 0, :3] + rng.uniform(-0.15, 0.15, (S, 3))
    return aos.reshape(S, 24), np.full(S, np.float32(0.12))


def _ref(aos, seg, steps):
    ref, grid = aos.copy(), None
    for _ in range(steps):
        grid = oracle.step32(oracle.Params(dt=1 / 64, damping=0.9, friction=0.05, hair_hair=True, grid_dim=16,
                                           grid_origin=(-0.5, -0.5, -0.5), grid_h=1 / 16, seg_length=seg), ref, 2, grid)
    ref = ref.reshape(-1, 3, 2, 4).copy()
    ref[:, 2] = 0
    return ref, grid.reshape(-1)


def test_box_counts(ctx):
    p = hairsim.step_params(damping=0.9, num_colliders=0, friction=0.05)
    data = [_groom(b, 100 + b) for b in BOXES]
    make = lambda d: ctx.groom(d[0], 2, seg_length=d[1], grid_dim=16, grid_origin=(-0.5, -0.5, -0.5), grid_h=1 / 16)  # noqa: E731
    alone, batch = [make(d) for d in data], [make(d) for d in data]
    try:
        for k in range(3):
            for g in alone:
                g.step(1 / 64, (k + 1) / 64, [], p)
            ctx.step_batch([(g, 1 / 64, (k + 1) / 64, [], p) for g in batch])
        for b, d, g, h in zip(BOXES, data, alone, batch):
            ref, grid = _ref(d[0], d[1], 3)
            for what, x in (("alone", g), ("batched", h)):
                out = x.read()[0].reshape(-1, 3, 2, 4).copy()
                out[:, 2] = 0
                assert_bitwise(out, ref, f"{b} boxes {what}", 2)
                assert np.array_equal(x.read_grid(), grid), (b, what)
    finally:
        for g in alone + batch:
            g.destroy()
