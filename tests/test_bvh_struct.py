"""drx_bvh filled by a caller that does not know its entry members: they are used only with their mark."""
import ctypes as C

import numpy as np
import pytest

from devil_ray_amd import _lib as L
from devil_ray_amd import synthetic as syn


def test_entry_mark():
    assert C.sizeof(L.DrxBVH) == 152 and L.DrxBVH.entry_mark.offset == 148
    v = L.DrxBVH()
    v.n_leaves, v.qnodes, v.entry_cells, v.entry_bits[:] = 33, 0x7F0000001000, 0x7F0000002000, [1, 2, 0]
    mark = L.lib().drx_bvh_entry_mark(C.byref(v))
    assert mark not in (0, 0xCDCDCDCD) and mark == L.lib().drx_bvh_entry_mark(C.byref(v))
    seen = {mark}
    for name, value in (("n_leaves", 34), ("qnodes", 0x7F0000003000), ("entry_cells", 0x7F0000003000)):
        w = L.DrxBVH.from_buffer_copy(v)
        setattr(w, name, value)
        seen.add(L.lib().drx_bvh_entry_mark(C.byref(w)))
    for bits in ([2, 1, 0], [1, 0, 2], [1, 2, 1]):
        w = L.DrxBVH.from_buffer_copy(v)
        w.entry_bits[:] = bits
        seen.add(L.lib().drx_bvh_entry_mark(C.byref(w)))
    assert len(seen) == 7
    for mesh_free in (L.DrxBVH(), L.DrxBVH.from_buffer_copy(b"\xcd" * C.sizeof(L.DrxBVH))):
        assert mesh_free.entry_mark != L.lib().drx_bvh_entry_mark(C.byref(mesh_free))


@pytest.mark.gpu
@pytest.mark.parametrize("fill", [0xCD, 0x05])
def test_entry_members_left_as_they_were(gpu, fill):
    """Every member but the entry ones set in memory that was not cleared: located as from the root, not refused."""
    m = gpu.UnstructuredMesh(syn.hex_mesh(5, 2, 0.05, 0.01, 3))
    bvh = m.get_bvh()
    pts = gpu.to_device(syn.query_points(5000, bvh.bounds, seed=5).reshape(-1))
    want = m.locate(pts).cpu().numpy()
    good, bad = bvh.view(), L.DrxBVH.from_buffer_copy(bytes([fill]) * C.sizeof(L.DrxBVH))
    for name, _ in L.DrxBVH._fields_:
        if not name.startswith("entry"):
            setattr(bad, name, getattr(good, name))
    out = gpu.to_device(np.zeros(4 * 5000, np.float32))
    mv, o = m.gf.view(), gpu.LocateOptions().c()
    rc = L.lib().drx_locate(C.byref(mv), C.byref(bad), C.c_void_p(pts.data_ptr()), 5000, C.c_void_p(out.data_ptr()), C.byref(o),
                            None)
    assert rc == 0, L.lib().drx_last_error()
    assert np.array_equal(out.cpu().numpy().view(np.uint8), want[: 16 * 5000])
