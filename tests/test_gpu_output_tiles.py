"""Device outputs at the edges of their LDS tiles: point counts that take each
tile width (32, 16 and 8 strand slots) and the longest strands, strand counts
of one slot, one short of and one past a tile, kept corrections (a third tile),
the draw record, and curve sample counts past the reciprocal divide.  Exports
equal the host read-back of the same state and its ref32 positions; curves the
oracle's restatement; bit for bit."""
import numpy as np
import pytest

import hairsim
import oracle
from hairsim import scenes
from helpers import assert_bitwise, gpu_params, make_gpu_groom, oracle_params

pytestmark = pytest.mark.gpu


def _stepped(ctx, wl, keep):
    g = wl.grooms[0]
    gpu = make_gpu_groom(ctx, wl, keep_corrections=keep)
    ref, grid = g.strands.copy(), None
    for k in range(2):
        gpu.step(wl.dt, float(wl.time(k)), [scenes.sphere_collider(wl.sphere(k))], gpu_params(wl, k))
        grid = oracle.step32(oracle_params(wl, k), ref, g.N, grid)
    return gpu, ref


@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("S,N", [(1, 2), (31, 52), (33, 53), (17, 107), (9, 108), (7, 256), (40, 256), (16500, 3), (140000, 2)])
def test_export_tiles(ctx, S, N, keep):
    wl = scenes.plain_100k(S=S, N=N, G=16)
    gpu, ref = _stepped(ctx, wl, keep)
    buf, ind = hairsim.DeviceBuffer(48 * S * N), hairsim.DeviceBuffer(16)
    try:
        buf.fill(0xFF)
        ind.fill(0xFF)
        gpu.export(buf, ind)
        ctx.sync()
        want = ref.reshape(S, 3, N, 4).copy()
        if not keep:
            want[:, 2] = 0
        assert_bitwise(buf.numpy(np.float32), want, f"export S={S} N={N}", N)
        assert tuple(ind.numpy(np.uint32)) == (S, 1, 0, 0)
    finally:
        buf.free()
        ind.free()
        gpu.destroy()


@pytest.mark.parametrize("S,N,M", [(33, 16, 8191), (33, 16, 8192), (140000, 2, 5), (3, 256, 5000), (1, 2, 2), (16500, 3, 4)])
def test_resample_tiles(ctx, S, N, M):
    wl = scenes.plain_100k(S=S, N=N, G=16)
    gpu, ref = _stepped(ctx, wl, False)
    out = hairsim.DeviceBuffer(16 * S * M)
    try:
        gpu.resample(M, out)
        ctx.sync()
        assert_bitwise(out.numpy(np.float32), oracle.resample32(ref, N, M).reshape(-1), f"resample S={S} N={N} M={M}")
    finally:
        out.free()
        gpu.destroy()
