"""When drx_locate sorts by itself, and what it does where the sort's memory or a launch fails (on the CPU, over
tests/fake_hip.c): without room for the sort the points are taken as they come, nothing is kept and no error is left; a
failing launch is reported.  And how it launches the points that it finds in order."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
N = 3 << 18   # enough points of order 3 for the sort

CHILD = r"""
import ctypes as C, json, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from devil_ray_amd import _lib as L
lib = L.lib()
get = lambda n, t=C.c_int: t.in_dll(fake, n)
get("fake_fail_malloc").value, get("fake_fail_launch").value = int(sys.argv[3]), int(sys.argv[4])
get("fake_first_copy").value = int(sys.argv[9])
n = int(sys.argv[5])
buf = C.create_string_buffer(64)
at = C.addressof(buf)
m, b, o = L.DrxMesh(), L.DrxBVH(), L.DrxLocateOpts()
order = int(sys.argv[8])
m.data, m.n_el, m.order, m.ncomp, m.stride = at, 1000, order, 3, lib.drx_mesh_stride(order, 3)
b.inner_nodes = b.leaf_pack = b.leaf_nodes = b.aabb_ids = b.subrefs = at
b.n_leaves = 33000 if order > 1 else 66000
b.bounds[:] = [0, 1, 0, 1, 0, 1]
o.coherent_order = int(sys.argv[6])
if int(sys.argv[7]):   # mixed orders
    m.elem_order = m.elem_offset = at
    m.order, m.stride = int(sys.argv[7]), 0
rc = lib.drx_locate(C.byref(m), C.byref(b), at, n, at, C.byref(o), None)
print(json.dumps([rc, (lib.drx_last_error() or b"").decode(), get("fake_mallocs").value, get("fake_launches").value,
                  get("fake_live", C.c_long).value, get("fake_grid").value]))
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", "-Wall", os.path.join(HERE, "fake_hip.c"), "-o", so])
    return so


def _run(fake, fail_malloc=-1, fail_launch=-1, n=N, coherent=0, mixed=0, order=3, far=1 << 20, grid=False):
    r = subprocess.run([sys.executable, "-c", CHILD, fake, os.path.dirname(HERE), str(fail_malloc), str(fail_launch), str(n),
                        str(coherent), str(mixed), str(order), str(far)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    out = json.loads(r.stdout.strip().splitlines()[-1])
    return out if grid else out[:5]


def test_no_room_for_the_sort(fake):
    rc, text, mallocs, launches, live = _run(fake)
    assert (rc, text) == (0, "") and mallocs == 7 and live >= 16 * N   # flags, the sort's six
    for k in range(1, mallocs):
        rc, text, got, fewer, live = _run(fake, fail_malloc=k)
        assert (rc, text) == (0, "") and got == k + 1 and fewer < launches and live < 4 * N, k
        # asked for, the sort is not left out
        rc, text, _, _, _ = _run(fake, fail_malloc=k, coherent=1)
        assert rc == 2 and "out of memory" in text, k


def test_failing_launch_is_reported(fake):
    _, _, _, launches, _ = _run(fake)
    assert launches > 8
    for k in range(launches):
        rc, text, _, _, _ = _run(fake, fail_launch=k)
        assert rc == 2 and "launch" in text, k


@pytest.mark.parametrize("order,least", [(4, 3 << 18), (3, 3 << 18), (2, 3 << 19)])
def test_mixed_orders_sort_from(fake, order, least):
    """A mesh of mixed orders whose largest is 4 is not taken for one of order 4: most of its elements may be of order 1."""
    assert _run(fake, n=least - 1, mixed=order)[2] == 1   # the flags alone
    assert _run(fake, n=least, mixed=order)[2] == 7


@pytest.mark.parametrize("order,n,chunked", [(1, 4 << 20, True), (1, 16 << 20, True), (2, 4 << 20, True), (2, 8 << 20, False),
                                             (3, 4 << 20, False), (4, 16 << 20, False)])
@pytest.mark.parametrize("far", [0, 1 << 20])
def test_cheap_elements_take_no_queue(fake, order, n, chunked, far):
    """The persistent launch's queue bounds points that cost little: order 1, and order 2 below 6 M points, go by chunks of
    256 whether they were found in order (far 0) or sorted."""
    rc, text, mallocs, _, _, grid = _run(fake, n=n, order=order, far=far, grid=True)
    assert (rc, text) == (0, "") and mallocs == (7 if far else 1)
    assert grid == n // 256 if chunked else grid < n // 256   # chunked: a wavefront for each; else the resident ones


def test_scans_of_a_sort(fake):
    """A radix pass counts the digits of 4,096 keys at a time; up to 10,240 counts are scanned by one launch, more by three."""
    one, last, three = (_run(fake, n=n, coherent=1)[3] for n in (8192, 40 * 4096, 40 * 4096 + 1))
    assert one == last and three == last + 2 * 3   # three passes
