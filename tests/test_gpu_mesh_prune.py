"""Pruned candidate lists of the mesh search: the nearest triangle of every
point, ties included, must still be listed.  Points all over a thin shell
around meshes of very different triangle and cell sizes (cells far larger and
far smaller than a triangle, a flat box with large coplanar faces and sharp
edges, a mesh far from the origin), one step each, bitwise against the
oracle's scan of every triangle."""
import numpy as np
import pytest

import hairsim
import oracle
from hairsim import scenes
from helpers import assert_bitwise

pytestmark = pytest.mark.gpu


def _box(n):
    """A unit box as n x n quads per face, two triangles each, outward."""
    verts, index, tris = [], {}, []

    def vid(p):
        k = tuple(np.round(p, 6))
        if k not in index:
            index[k] = len(verts)
            verts.append(p)
        return index[k]

    for axis in range(3):
        for side in (-0.5, 0.5):
            u, v = (axis + 1) % 3, (axis + 2) % 3
            for i in range(n):
                for j in range(n):
                    q = []
                    for a, b in ((0, 0), (1, 0), (1, 1), (0, 1)):
                        p = np.zeros(3)
                        p[axis], p[u], p[v] = side, (i + a) / n - 0.5, (j + b) / n - 0.5
                        q.append(vid(p))
                    if side < 0:
                        q = q[::-1]
                    tris += [(q[0], q[1], q[2]), (q[0], q[2], q[3])]
    return np.array(verts, np.float32), np.array(tris, np.uint32)


MESHES = {
    "coarse sphere, fine cells": (lambda: scenes.icosphere(1), (60, 64, 60), 0.08),
    "fine sphere, coarse cells": (lambda: scenes.icosphere(4), (7, 9, 8), 0.05),
    "box, fine cells": (lambda: _box(3), (48, 50, 52), 0.1),
    "box, one cell": (lambda: _box(4), (1, 1, 1), 0.1),
    "sphere far from the origin": (lambda: tuple(a + np.float32([40, -25, 60]) if a.dtype == np.float32 else a
                                                 for a in scenes.icosphere(3)), (40, 40, 40), 0.07),
}


@pytest.mark.parametrize("name", list(MESHES))
def test_nearest_is_listed(ctx, name):
    make, grid, margin = MESHES[name]
    V, T = make()
    rng = np.random.default_rng(5)
    S, N = 3000, 2
    # points just inside and around random surface points, vertices and edges
    t = T[rng.integers(0, len(T), S)]
    w = rng.dirichlet((0.6, 0.6, 0.6), S)
    w[: S // 6] = np.round(w[: S // 6])  # at vertices
    on = np.einsum("sk,skc->sc", w, V[t].astype(np.float64))
    centre = V.mean(0).astype(np.float64)
    x = on + (centre - on) * rng.uniform(-0.05, 1.2 * margin, (S, 1))
    aos = np.zeros((S, 3, N, 4), np.float32)
    aos[:, 0, :, 3] = 1
    aos[:, 0, 0, :3] = x - 0.1
    aos[:, 0, 1, :3] = x
    mid = ctx.mesh(V, T, grid_dim=grid, margin=margin)
    gr = ctx.groom(aos.reshape(-1), N, strand_length=0.2)
    try:
        gr.step(1 / 60, 1 / 60, [], hairsim.step_params(num_colliders=0, hair_hair=False, mesh_id=mid))
        out = gr.read()[0].reshape(S, 3, N, 4).copy()
    finally:
        gr.destroy()
        ctx.mesh_destroy(mid)
    p = dict(dt=1 / 60, damping=0.998, hair_hair=False, seg_length=np.full(S, np.float32(0.2)), colliders=None)
    ref = aos.copy().reshape(S, 12 * N)
    oracle.step32(oracle.Params(mesh=oracle.mesh_prepare(V, T), mesh_margin=margin, **p), ref, N, None)
    free = aos.copy().reshape(S, 12 * N)
    oracle.step32(oracle.Params(**p), free, N, None)
    hit = (ref != free).any(1).mean()
    print(f"{name}: {hit:.2f} of the strands in contact", flush=True)
    assert hit > 0.2
    ref = ref.reshape(S, 3, N, 4)
    out[:, 2] = 0
    ref[:, 2] = 0
    assert_bitwise(out, ref, name, N)
