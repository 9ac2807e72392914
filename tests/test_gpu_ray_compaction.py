"""Ray and partial compaction and the tile order against NumPy, where the number of launches changes: one tile, a partial
block, the last tile count of the one-block sort and the first beyond it, counts that are added up by the blocks and
counts that are scanned first."""
import numpy as np
import pytest

from devil_ray_amd import synthetic as syn
from devil_ray_amd.api import RAY_DTYPE
from test_gpu_parity import _np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (8, 8), (33, 31), (321, 255), (1024, 1024), (1032, 1024), (2056, 2048)])
@pytest.mark.parametrize("miss", [False, True])
def test_rays_kept_and_ordered(gpu, orc, w, h, miss):
    print(f"[ray compaction] {w}x{h} miss={miss}", flush=True)
    cam = gpu.Camera(w, h, 40.0, pos=(0.5, 0.6, 2.4 if miss else 1.2), look_at=(0.5, 0.5, 0.5))
    rays = cam.create_rays()
    bounds = np.array([0, 1, 0, 1, 0, 1], np.float32)
    act, n = gpu.remove_missed_rays(rays, bounds)
    host = _np(rays, np.uint8).view(RAY_DTYPE)
    ref = orc.remove_missed_rays(host, bounds)
    got = _np(act, np.uint8)[: n * RAY_DTYPE.itemsize].view(RAY_DTYPE)
    assert n == len(ref) and np.array_equal(got["pixel_id"], ref["pixel_id"])
    assert np.array_equal(got["near"], ref["near"]) and np.array_equal(got["far"], ref["far"])
    assert not miss or w * h < 2000 or 0 < n < w * h
    order = _np(gpu.ray_tile_order(act, n, w, h))[:n]
    # tile by its longest segment, descending, then by index; inside a tile by row, then column
    pid = got["pixel_id"].astype(np.int64)
    tile = (pid // w // 8) * ((w + 7) // 8) + (pid % w) // 8
    longest = np.full(((w + 7) // 8) * ((h + 7) // 8), -1.0, np.float32)
    np.maximum.at(longest, tile, np.maximum(got["far"] - got["near"], 0))
    assert np.array_equal(order, np.lexsort((pid, tile, -longest[tile])))


@pytest.mark.parametrize("w,h", [(37, 29), (1032, 1024)])
def test_partials_kept_in_ray_order(gpu, w, h):
    print(f"[partial compaction] {w}x{h}", flush=True)
    mesh = syn.hex_mesh(4, 1, 0.05, 0.01, 3)
    vol = gpu.Volume(gpu.UnstructuredMesh(mesh), gpu.UnstructuredField(mesh))
    vol.use_lighting = False
    vol.samples(24)
    vol.table.add_alpha(0.0, 0.3)
    act, n = gpu.remove_missed_rays(gpu.Camera(w, h, 40.0, pos=(0.5, 0.6, 1.2), look_at=(0.5, 0.5, 0.5)).create_rays(),
                                    vol.mesh.bounds())
    parts, cnt = vol.integrate(None, active=(act, n))
    whole = _np(parts, np.uint8)[: cnt * 24]
    pieces, size, step = [], RAY_DTYPE.itemsize, (n + 3) // 4
    for lo in range(0, n, step):
        k = min(step, n - lo)
        p, c = vol.integrate(None, active=(act[lo * size : (lo + k) * size].clone(), k))
        pieces.append(_np(p, np.uint8)[: c * 24])
    assert cnt > n // 2 and np.array_equal(whole, np.concatenate(pieces))
