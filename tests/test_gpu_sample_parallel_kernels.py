"""Both sample-parallel kernels against one lane per ray, each on frames that it takes (drx_integrate_stats.binned says
which ran): the same partials and located, Newton, candidate and polished counts."""
import ctypes as C

import numpy as np
import pytest

from devil_ray_amd import _lib as L
from devil_ray_amd import synthetic as syn
from test_gpu_parity import _np, _slab_stack


def test_stats_layout():
    assert L.DrxIntegrateStats.binned.offset == 44 and C.sizeof(L.DrxIntegrateStats) == 48


def _compare(gpu, mesh, rays, side, samples, lit, polish, fp64, binned, lights=None, alpha=0.3):
    vol = gpu.Volume(gpu.UnstructuredMesh(mesh), gpu.UnstructuredField(mesh, fp64=fp64))
    vol.use_lighting = lit
    vol.samples(samples)
    vol.table = gpu.ColorTable()
    vol.table.add_point(0.0, (0.2, 0.4, 0.9))
    vol.table.add_point(1.0, (1.0, 0.3, 0.0))
    vol.table.add_alpha(0.0, alpha)
    got = {}
    for launch in (1, 3):
        vol.opts = gpu.LocateOptions(launch=launch, traversal=3, fp64_polish=polish, cond_threshold=1.0 if polish else 1e4)
        parts, n = vol.integrate(rays, tile_width=side, tile_height=side, lights=lights)
        st = vol.last_stats
        assert (st.walk, st.binned) == ((0, 0) if launch == 1 else (5, binned))
        got[launch] = ((st.located_samples, st.newton_steps, st.candidates, st.polished), _np(parts, np.uint8)[: n * 24].copy())
    assert got[1][0][0] > 0 and (not polish or got[1][0][3] > 0)
    assert got[1][0] == got[3][0]
    assert np.array_equal(got[1][1], got[3][1])
    return got[3][1]


# Grouped by element: fine meshes, seen along an axis, obliquely (wavefronts whose leaves outgrow the list) and from inside.
FINE = [
    ("p1_n16", lambda: syn.hex_mesh(16, 1, 0.05, 0.01, 3), (0.5, 0.5, 3.0), 240, 300, False, False, False),
    ("p2_n14_fp64_field", lambda: syn.hex_mesh(14, 2, 0.05, 0.01, 5, keep_field64=True), (2.2, 2.0, 2.3), 330, 300, False, False,
     True),
    ("p3_n12_lit", lambda: syn.hex_mesh(12, 3, 0.1, 0.01, 4), (-1.4, 1.9, 2.0), 300, 220, True, False, False),
    ("p4_n10_polish", lambda: syn.hex_mesh(10, 4, 0.2, 0.01, 6), (2.2, 2.0, 2.3), 200, 130, False, True, False),
    ("mixed_n10", lambda: syn.mixed_hex_mesh(10, 0.1, 0.01, 7), (2.2, 2.0, 2.3), 210, 150, False, False, False),
    ("p3_n12_inside", lambda: syn.hex_mesh(12, 3, 0.1, 0.01, 8), (0.52, 0.48, 0.55), 120, 160, False, True, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,pos,side,samples,lit,polish,fp64", FINE, ids=[c[0] for c in FINE])
def test_grouped_on_fine_meshes(gpu, name, make, pos, side, samples, lit, polish, fp64):
    print(f"[grouped] {name}", flush=True)
    cam = gpu.Camera(side, side, 45.0, pos=pos, look_at=(0.5, 0.5, 0.5))
    _compare(gpu, make(), cam.create_rays(), side, samples, lit, polish, fp64, 1, [gpu.default_light(cam)])


# A sample per lane: fewer than 32 active rays per element column.
SPARSE = [("p1", lambda: syn.hex_mesh(12, 1, 0.05, 0.01, 11, keep_field64=True)),
          ("p2", lambda: syn.hex_mesh(12, 2, 0.05, 0.01, 1, keep_field64=True)),
          ("p3", lambda: syn.hex_mesh(11, 3, 0.1, 0.01, 2, keep_field64=True)),
          ("p4", lambda: syn.hex_mesh(10, 4, 0.25, 0.01, 3, keep_field64=True)),
          ("mixed", lambda: syn.mixed_hex_mesh(11, 0.15, 0.05, 5))]


@pytest.mark.gpu
@pytest.mark.parametrize("name,make", SPARSE, ids=[c[0] for c in SPARSE])
def test_sample_per_lane(gpu, name, make):
    mesh = make()
    cam = gpu.Camera(40, 40, 45.0, pos=(0.5, 0.6, 2.5), look_at=(0.5, 0.5, 0.5))
    for lit, polish, fp64, samples in ((False, False, False, 96), (True, False, False, 96), (False, True, False, 96),
                                       (True, True, False, 64), (False, False, True, 96), (False, True, True, 70),
                                       (False, False, False, 5)):
        if fp64 and mesh.field64 is None:
            continue
        print(f"[sample per lane] {name} lit={lit} polish={polish} fp64={fp64} samples={samples}", flush=True)
        _compare(gpu, mesh, cam.create_rays(), 40, samples, lit, polish, fp64, 0, [gpu.default_light(cam)])


@pytest.mark.gpu
def test_sample_per_lane_partial_limit(gpu):
    rays = syn.orthographic_rays(24, 24)
    parts = _compare(gpu, _slab_stack(), gpu.as_bytes(rays), 24, 200, False, False, False, 0, alpha=0.02)
    per_ray = np.bincount(parts.view(syn.PARTIAL_DTYPE)["pixel_id"], minlength=24 * 24)
    assert (per_ray == 5).sum() > 288 and per_ray.max() == 5


@pytest.mark.gpu
@pytest.mark.parametrize("p", [1, 2, 3, 4, 0])
def test_coarse_march_per_lane(gpu, p):
    """Steps as long as an element: the form that ran before candidates were grouped, in small and in large frames."""
    n = 14 if p < 4 else 13
    mesh = syn.hex_mesh(n, p, 0.05, 0.01, 3) if p else syn.mixed_hex_mesh(n, 0.1, 0.01, 3)
    cam = gpu.Camera(200, 200, 45.0, pos=(2.2, 2.0, 2.3), look_at=(0.5, 0.5, 0.5))
    _compare(gpu, mesh, cam.create_rays(), 200, 8, False, False, False, 0)
    vol = gpu.Volume(gpu.UnstructuredMesh(mesh), gpu.UnstructuredField(mesh))
    vol.use_lighting = False
    side = 640
    for samples, want in ((8, (0, 0)), (400, (5, 1))):
        vol.samples(samples)
        vol.integrate(gpu.Camera(side, side, 60.0, pos=(0.5, 0.5, 0.95), look_at=(0.5, 0.5, 0.0)).create_rays(), tile_width=side,
                      tile_height=side)
        assert (vol.last_stats.walk, vol.last_stats.binned) == want, samples


@pytest.mark.gpu
@pytest.mark.parametrize("n,p,side", [(12, 3, 304), (14, 2, 640)])   # whole tiles
def test_rays_in_no_order_per_lane(gpu, n, p, side):
    """The form is chosen by how the rays lie in processing order: grouped in tile order; a sample (small frame) or a ray
    (more than 300 active rays per SIMD) per lane for the same rays shuffled.  The partials of a ray are the same."""
    mesh = syn.hex_mesh(n, p, 0.1, 0.01, 4)
    m = gpu.UnstructuredMesh(mesh)
    vol = gpu.Volume(m, gpu.UnstructuredField(mesh))
    vol.use_lighting = False
    vol.samples(200)
    vol.table = gpu.ColorTable()
    vol.table.add_alpha(0.0, 0.3)
    cam = gpu.Camera(side, side, 60.0, pos=(0.5, 0.5, 0.95), look_at=(0.4, 0.45, 0.0))
    act, k = gpu.remove_missed_rays(cam.create_rays(), m.bounds())
    rays = _np(act, np.uint8)[: k * 36].reshape(k, 36)
    perm = np.random.default_rng(3).permutation(k)
    parts, cnt = vol.integrate(None, tile_width=side, tile_height=side, active=(act, k))
    assert (vol.last_stats.walk, vol.last_stats.binned) == (5, 1)
    counts = (vol.last_stats.newton_steps, vol.last_stats.candidates)
    a = _np(parts, np.uint8)[: cnt * 24].view(syn.PARTIAL_DTYPE)
    parts, cnt2 = vol.integrate(None, active=(gpu.as_bytes(rays[perm].copy()), k))
    assert (vol.last_stats.walk, vol.last_stats.binned) == (5 if side < 500 else 0, 0)
    assert counts == (vol.last_stats.newton_steps, vol.last_stats.candidates)
    b = _np(parts, np.uint8)[: cnt2 * 24].view(syn.PARTIAL_DTYPE)
    assert cnt == cnt2
    assert np.array_equal(np.sort(a, order=["pixel_id", "depth"]).view(np.uint8), np.sort(b, order=["pixel_id", "depth"]).view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("opacity,grouped", [(0.10, 1), (0.13, 0), (1.0, 0)])
@pytest.mark.parametrize("lit", [False, True])
def test_opaque_tables_per_lane(gpu, opacity, grouped, lit):
    """A colour table with which a ray can end within 24 samples (opacity per sample 1 - 0.05^(1/24) = 0.117) keeps the form
    that works a sample, or in frames of more than 300 active rays per SIMD a ray, per lane."""
    mesh = syn.hex_mesh(14, 2, 0.05, 0.01, 3)
    alpha = 1.0 - (1.0 - opacity) ** 20.0   # the table is corrected by 10 / samples
    cam = gpu.Camera(120, 120, 60.0, pos=(0.5, 0.5, 0.95), look_at=(0.5, 0.5, 0.0))
    _compare(gpu, mesh, cam.create_rays(), 120, 200, lit, False, False, grouped, [gpu.default_light(cam)], alpha)
    vol = gpu.Volume(gpu.UnstructuredMesh(mesh), gpu.UnstructuredField(mesh))
    vol.use_lighting = lit
    vol.samples(200)
    vol.table = gpu.ColorTable()
    vol.table.add_alpha(0.0, alpha)
    cam = gpu.Camera(640, 640, 60.0, pos=(0.5, 0.5, 0.95), look_at=(0.5, 0.5, 0.0))
    vol.integrate(cam.create_rays(), tile_width=640, tile_height=640, lights=[gpu.default_light(cam)])
    assert (vol.last_stats.walk, vol.last_stats.binned) == ((5, 1) if grouped else (0, 0))


@pytest.mark.gpu
def test_many_candidates_counted(gpu):
    """2,200 thin slabs on the diagonal of one small box: a sample beside their plane is in more than 4,095 leaf boxes and
    in no element. The frame is left to the form that counts them all."""
    slab = syn.box_net((0.0, 0.0, -1e-3), (0.14, 0.1, 1e-3), 1)
    c = np.sqrt(0.5)
    slab = slab @ np.array([[c, 0.0, c], [0.0, 1.0, 0.0], [-c, 0.0, c]]) + [0.45, 0.45, 0.45]
    nets = [slab] * 2200 + [syn.box_net((x, y, z), (x + 0.1, y + 0.4, z + 0.1), 1)
                            for x in (0.0, 0.9) for y in (0.0, 0.6) for z in (0.0, 0.9)]
    field = np.random.default_rng(1).uniform(0, 1, (len(nets), 8))
    mesh = syn.elements_from_nets(np.stack(nets), 1, field=field)
    side = 96
    g = (np.arange(side) + 0.5) / side
    rays = syn.orthographic_rays(side, side)
    rays["orig"][:, 0], rays["orig"][:, 1], rays["orig"][:, 2] = np.tile(g, side), -0.5, np.repeat(g, side)
    rays["dir"] = (1e-7, 1.0, 1e-7)
    _compare(gpu, mesh, gpu.as_bytes(rays), side, 160, False, False, False, 0, alpha=0.2)


@pytest.mark.gpu
@pytest.mark.parametrize("p,shear", [(2, 0.0), (2, 8.0), (3, 5.0)])
def test_sheared_elements_per_lane(gpu, p, shear):
    """Elements sheared over several of their widths: their boxes overlap, some points have many candidates, and the form
    that goes round until all are settled is not taken."""
    mesh = syn.hex_mesh(8, p, 0.02, 0.01, 3)
    mesh.values[:, 0] += np.float32(shear) * mesh.values[:, 2]
    c = 0.5 * (1.0 + shear)
    cam = gpu.Camera(200, 200, 45.0, pos=(c, 0.5, 2.5 + shear), look_at=(c, 0.5, 0.5))
    _compare(gpu, mesh, cam.create_rays(), 200, 300, False, False, False, 0 if shear else 1)
