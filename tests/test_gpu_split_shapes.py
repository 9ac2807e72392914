"""The element split on elements that its level-parallel form treats differently: equal measures (the largest-first
rule's ties), zero volumes, measures that differ so much that the rule runs down one corner of the element, tangled
nets.  Boxes, SubRefs and ids are the oracle's bit for bit."""
import numpy as np
import pytest

from devil_ray_amd import synthetic as syn
from test_gpu_parity import _np

pytestmark = pytest.mark.gpu


def _nets(p):
    """One net per shape, as (p+1)^3 x 3 float64."""
    rng = np.random.default_rng(70 + p)
    cube = syn.box_net((0.25, 0.5, 0.75), (1.25, 1.5, 1.75), p)
    u = (cube - cube[0]) / (cube[-1] - cube[0])
    flat = cube.copy()
    flat[:, 2] = 0.5
    return [cube,                                                      # every level's volumes tie
            syn.box_net((0.1, 0.2, 0.3), (8.1, 0.7, 0.4), p),          # ties with unequal extents
            flat, np.full_like(cube, 0.5),                             # zero volume, zero surface
            1.0 + u ** 6, 1.0 + np.exp2(18.0 * u), 1.0 + u * [1e-6, 1.0, 1e6],   # graded: deep paths
            1.0 + np.exp2(18.0 * (1.0 - u)),
            cube + rng.uniform(-0.02, 0.02, cube.shape), cube + rng.uniform(-0.3, 0.3, cube.shape),
            rng.uniform(1.0, 2.0, cube.shape)]                         # tangled


@pytest.mark.parametrize("p", [1, 2, 3, 4, 5, 8])
def test_split_shapes_bit_exact(gpu, orc, p):
    print(f"[split shapes] order {p}", flush=True)
    mesh = syn.elements_from_nets(np.stack(_nets(p)), p)
    aabbs, prims, subrefs = gpu.UnstructuredMesh(mesh).split_elements()
    oa, op, osr = orc.split_elements(mesh)
    assert np.array_equal(_np(prims), op)
    assert np.array_equal(_np(subrefs).reshape(-1, 6).view(np.uint32), osr.view(np.uint32))
    assert np.array_equal(_np(aabbs).reshape(-1, 6).view(np.uint32), oa.view(np.uint32))
