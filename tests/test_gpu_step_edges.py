"""The step kernel where its split of a segment's points over a strand's
threads has edges: strands that end on a segment's or a thread's last point,
one past it, and one before it, for every tile shape; workgroups with a single
strand or one short of full; boxes of many splat windows and of more than the
kernel splats through windows.  Bitwise against ref32."""
import pytest

import hairsim
import oracle
from hairsim import scenes
from helpers import assert_bitwise, gpu_params, make_gpu_groom, oracle_params, run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strands,points", hairsim.TILE_SHAPES)
def test_points_at_segment_and_thread_edges(ctx, strands, points):
    """1 + k points for k around multiples of a thread's share and of the
    segment (the last strand point has no successor to hand its velocity to)."""
    per = {(128, 16): 4, (256, 8): 4, (256, 12): 6}[(strands, points)]
    ctx.set_tile(2048, 2048, 1, strands, points)
    try:
        for k in sorted({1, 2, per - 1, per, per + 1, points - 1, points, points + 1, 2 * points, 2 * points + 1}):
            for S in (1, strands - 1, strands + 1):
                print(f"shape {strands}x{points} N {1 + k} S {S}", flush=True)
                run_parity(ctx, scenes.plain_100k(S=S, N=1 + k, G=16), 3)
    finally:
        ctx.set_tile(2048, 2048, 1)


@pytest.mark.parametrize("strands,points", hairsim.TILE_SHAPES)
@pytest.mark.parametrize("window", [64, 512])
def test_boxes_of_many_windows(ctx, strands, points, window):
    """300 strands over the whole hemisphere on a 48^3 grid: boxes of about
    30^3 voxels, hundreds of 64-cell windows (beyond the limit: device atomics
    into the overflow grid, which is not a fallback) or tens of 512-cell ones."""
    wl = scenes.plain_100k(S=300, N=20, G=48)
    ctx.set_tile(2048, window, 0, strands, points)
    try:
        run_parity(ctx, wl, 4)
        g = wl.grooms[0]
        gr = ctx.groom(g.strands, g.N, seg_length=g.seg, wind_noise=g.noise, grid_dim=g.grid_dim,
                       grid_origin=g.grid_origin, grid_h=g.grid_h)
        gr.step(wl.dt, float(wl.time(0)), [scenes.sphere_collider(wl.sphere(0))],
                hairsim.step_params(num_colliders=1, sphere_radius=0.3))
        assert gr.grid_work()["deferred"] > 0
        gr.destroy()
    finally:
        ctx.set_tile(2048, 2048, 1)


def test_corrections_and_plain_steps_at_edges(ctx):
    """Kept corrections, and steps without the grid (no splat, no gather)."""
    wl = scenes.plain_100k(S=130, N=17, G=16)
    run_parity(ctx, wl, 3, keep_corrections=True)
    for N in (2, 5, 9, 10, 16, 17, 18, 33):  # up to 9 points take the 256 x 8 kernel whatever the tile
        run_parity(ctx, scenes.plain_1k(S=130, N=N), 3, keep_corrections=True)


@pytest.mark.parametrize("N", [2, 9, 10])
def test_grid_switched_on_and_off(ctx, N):
    """Steps with and without the grid in turn: the latter may run another
    shape, which must not be taken for the layout of the last splat's boxes."""
    wl = scenes.plain_100k(S=300, N=N, G=16)
    g = wl.grooms[0]
    gpu = make_gpu_groom(ctx, wl)
    ref, grid = g.strands.copy(), None
    try:
        for k, on in enumerate([True, False, False, True, True, False, True]):
            c = [scenes.sphere_collider(wl.sphere(k))]
            gpu.step(wl.dt, float(wl.time(k)), c, gpu_params(wl, k, hair_hair=on))
            grid = oracle.step32(oracle_params(wl, k, hair_hair=on), ref, N, grid)
        out = gpu.read()[0].reshape(-1, 3, N, 4).copy()
        want = ref.reshape(-1, 3, N, 4).copy()
        out[:, 2] = 0
        want[:, 2] = 0
        assert_bitwise(out, want, f"N={N}", N)
    finally:
        gpu.destroy()
