"""Large batches that drx_locate sorts itself against drx_locate_noalloc, which never does: the same locations, Newton
steps, candidates and polished flags, for points in no order, in order, outside the mesh and not finite."""
import ctypes as C

import numpy as np
import pytest
import torch

from devil_ray_amd import _lib as L
from devil_ray_amd import synthetic as syn
from devil_ray_amd.api import _ptr, _stream

pytestmark = pytest.mark.gpu


def _run(fn, m, pts, opts):
    n = pts.numel() // 3
    out = torch.zeros(n * 16, dtype=torch.uint8, device=pts.device)
    extra = [torch.zeros(n, dtype=torch.int32, device=pts.device) for _ in range(3)]
    o, mv, bv = opts.c(*extra), m.gf.view(), m.get_bvh().view()
    assert fn(C.byref(mv), C.byref(bv), _ptr(pts), n, _ptr(out), C.byref(o), _stream()) == 0
    return [out.cpu().numpy()] + [e.cpu().numpy() for e in extra]


# mesh, points, their order, FP64 polish: at the least number of points and one below it, for each order's rule
CASES = [
    ("p1", lambda: syn.hex_mesh(14, 1, 0.1, 0.01, 3), 3 << 19, "random", False),
    ("p1_small_mesh", lambda: syn.hex_mesh(6, 1, 0.1, 0.01, 3), 3 << 19, "random", False),
    ("p2", lambda: syn.hex_mesh(8, 2, 0.1, 0.01, 3), (3 << 19) + 77, "random", True),
    ("p3", lambda: syn.hex_mesh(8, 3, 0.1, 0.01, 3), 3 << 18, "random", False),
    ("p3_below", lambda: syn.hex_mesh(8, 3, 0.1, 0.01, 3), (3 << 18) - 1, "random", False),
    ("p3_sorted", lambda: syn.hex_mesh(8, 3, 0.1, 0.01, 3), 3 << 18, "sorted", False),
    ("p3_outside", lambda: syn.hex_mesh(8, 3, 0.1, 0.01, 3), 3 << 18, "outside", False),
    ("p4", lambda: syn.hex_mesh(7, 4, 0.1, 0.01, 3), (3 << 17) + 1, "random", True),
    ("mixed", lambda: syn.mixed_hex_mesh(8, 0.1, 0.02, 4), 3 << 17, "random", True),
    ("p5", lambda: syn.hex_mesh(7, 5, 0.05, 0.01, 3), 3 << 17, "random", False),
]


@pytest.mark.parametrize("name,make,n,kind,polish", CASES, ids=[c[0] for c in CASES])
def test_sorted_by_size_identical(gpu, name, make, n, kind, polish):
    print(f"[locate order] {name} n={n}", flush=True)
    m = gpu.UnstructuredMesh(make())
    rng = np.random.default_rng(n)
    pts = rng.uniform(-0.05, 1.05, (n, 3)).astype(np.float32)
    if kind == "sorted":
        pts = pts[np.lexsort(((pts[:, 0] * 64).astype(int), (pts[:, 1] * 64).astype(int), (pts[:, 2] * 64).astype(int)))]
    if kind == "outside":
        pts[rng.integers(0, n, n // 2)] += 7.0
        pts[rng.integers(0, n, 999)] = np.nan
        pts[rng.integers(0, n, 999)] = np.inf
    d = gpu.to_device(pts.reshape(-1))
    opts = gpu.LocateOptions(fp64_polish=polish, cond_threshold=10.0)
    got = _run(L.lib().drx_locate, m, d, opts)
    ref = _run(L.lib().drx_locate_noalloc, m, d, opts)
    assert (ref[0].view(np.int32).reshape(n, 4)[:, 0] >= 0).any()
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)
