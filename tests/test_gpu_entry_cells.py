"""Walks that start from entry cells (drx_bvh_entry_cells) against walks from the root: the same cells, reference
points (bitwise), Newton steps and candidate counts, for every shape of cell grid, on box faces and outside."""
import ctypes as C

import numpy as np
import pytest
import torch

from devil_ray_amd import synthetic as syn
from devil_ray_amd.synthetic import LOCATION_DTYPE
from test_gpu_parity import _np

pytestmark = pytest.mark.gpu


def _flat():
    m = syn.hex_mesh(3, 1, 0.0, 0.0, 1)
    m.values[:, 2] = 0.5   # zero extent along z
    return m


def _thin():
    m = syn.hex_mesh(4, 2, 0.05, 0.01, 5)
    m.values *= np.array([100.0, 1.0, 0.01], np.float32)
    return m


MESHES = [("p1_n1", lambda: syn.hex_mesh(1, 1, 0.0, 0.0, 1)), ("p3_n5", lambda: syn.hex_mesh(5, 3, 0.1, 0.01, 2)),
          ("p4_n3", lambda: syn.hex_mesh(3, 4, 0.2, 0.01, 3)), ("mixed_n4", lambda: syn.mixed_hex_mesh(4, 0.1, 0.01, 4)),
          ("thin", _thin), ("flat", _flat)]


@pytest.mark.parametrize("name,make", MESHES, ids=[m[0] for m in MESHES])
def test_entry_cells_same_candidates(gpu, name, make):
    print(f"[entry cells] {name}", flush=True)
    m = gpu.UnstructuredMesh(make())
    bvh = m.get_bvh()
    pts = syn.query_points(20000, bvh.bounds, seed=7)
    corners = _np(bvh.leaf_boxes).reshape(-1, 8)[:, :6].reshape(-1, 3)[:4000]   # on the leaf boxes' faces
    b = bvh.bounds
    odd = [(np.nan, 0.5, 0.5), (0.5, np.nan, np.nan), (np.inf, 0.5, 0.5), (-np.inf, 0, 0), (1e30, 0.5, 0.5),
           (b[0], b[2], b[4]), (b[1], b[3], b[5]), (np.nextafter(b[1], np.float32(np.inf)), b[3], b[5]), (0.0, -0.0, 0.0)]
    pts = np.concatenate([pts, corners, np.array(odd, np.float32)]).astype(np.float32)
    d = gpu.to_device(pts.reshape(-1))

    def run():
        loc, steps, cands = m.locate(d, gpu.LocateOptions(traversal=3), stats=True)
        l = _np(loc, LOCATION_DTYPE)
        return l["cell"].copy(), l["ref"].view(np.uint32).copy(), _np(steps), _np(cands)

    auto, bits = bvh.entry_cells, bvh.entry_bits.copy()
    assert auto is not None and int(bits.sum()) <= 24
    got = {"auto": run()}
    for shape in ((0, 0, 0), (3, 0, 5), (6, 6, 6), (0, 14, 1), (2, 9, 6)):
        out = torch.empty(4 << sum(shape), dtype=torch.int32, device="cuda")
        bvh.entry_bits = np.array(shape, np.int32)
        v = bvh.view()
        gpu.L.check(gpu.L.lib().drx_bvh_entry_cells(C.byref(v), bvh.entry_bits.ctypes.data, C.c_void_p(out.data_ptr()),
                                                    None), "drx_bvh_entry_cells")
        torch.cuda.synchronize()
        bvh.entry_cells = out
        got[shape] = run()
    bvh.entry_cells = None
    ref = run()
    bvh.entry_cells, bvh.entry_bits = auto, bits
    for shape, g in got.items():
        for a, r in zip(g, ref):
            assert np.array_equal(a, r), shape
