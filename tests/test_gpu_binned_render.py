"""The sample-parallel render that bins candidates by element against one lane per ray: the same partials and located,
Newton, candidate and polished counts, where its leaf lists, walks and rounds differ most."""
import numpy as np
import pytest

from devil_ray_amd import synthetic as syn
from test_gpu_parity import _np

pytestmark = pytest.mark.gpu


def _soup():
    """Overlapping elements: points lie in many boxes and several elements."""
    rng = np.random.default_rng(5)
    nets = []
    for _ in range(24):
        lo = rng.uniform(0.0, 0.6, 3)
        nets.append(syn.box_net(lo, lo + rng.uniform(0.2, 0.4, 3), 2) + rng.uniform(-0.02, 0.02, (27, 3)))
    return syn.elements_from_nets(np.stack(nets), 2, field=rng.uniform(0, 1, (24, 27)))


# mesh, camera position, frame, samples, lit, FP64 polish, compact nodes, entry cells
CASES = [
    ("oblique_p1_n16", lambda: syn.hex_mesh(16, 1, 0.05, 0.01, 3), (2.2, 2.0, 2.3), 131, 200, False, False, True, True),
    ("oblique_p3_n12", lambda: syn.hex_mesh(12, 3, 0.15, 0.01, 4), (-1.4, 1.9, 2.0), 101, 150, True, False, True, True),
    ("soup", _soup, (0.5, 0.6, 2.6), 67, 90, False, True, True, True),
    ("soup_lit", _soup, (2.0, 1.8, 1.9), 60, 90, True, False, True, False),
    ("no_compact_nodes", lambda: syn.hex_mesh(3, 2, 0.05, 0.01, 6), (0.5, 0.5, 2.5), 50, 64, False, False, False, False),
    ("mixed_inside", lambda: syn.mixed_hex_mesh(4, 0.1, 0.01, 7), (0.52, 0.48, 0.55), 65, 70, False, True, True, True),
]


@pytest.mark.parametrize("name,make,pos,side,samples,lit,polish,compact,cells", CASES, ids=[c[0] for c in CASES])
def test_binned_render_identical(gpu, name, make, pos, side, samples, lit, polish, compact, cells):
    print(f"[binned render] {name}", flush=True)
    mesh = make()
    m = gpu.UnstructuredMesh(mesh)
    bvh = m.get_bvh()
    bvh.use_qnodes = compact
    if not cells:
        bvh.entry_cells = None
    cam = gpu.Camera(side, side, 45.0, pos=pos, look_at=(0.5, 0.5, 0.5))
    vol = gpu.Volume(m, gpu.UnstructuredField(mesh))
    vol.use_lighting = lit
    vol.samples(samples)
    vol.table.add_alpha(0.0, 0.3)
    lights = [gpu.default_light(cam)]
    got = {}
    for launch in (1, 3):
        vol.opts = gpu.LocateOptions(launch=launch, traversal=3, fp64_polish=polish, cond_threshold=1.0 if polish else 1e4)
        parts, n = vol.integrate(cam.create_rays(), tile_width=side, tile_height=side, lights=lights)
        st = vol.last_stats
        assert st.walk == (0 if launch == 1 else 5)
        got[launch] = (n, (st.located_samples, st.newton_steps, st.candidates, st.polished),
                       _np(parts, np.uint8)[: n * 24].copy())
    assert got[1][1][0] > 0 and got[1][1][2] >= got[1][1][0]
    assert got[1][:2] == got[3][:2]
    assert np.array_equal(got[1][2], got[3][2])
