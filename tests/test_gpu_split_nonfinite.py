"""The element split of nets with NaN, infinite and huge control points: its largest-first rule meets measures that are
NaN, infinite or empty, which its ranks leave to the rule's own order.  Boxes, SubRefs and ids are the oracle's bit for bit.
(A NaN at the first control point is left out: dray's running min / max keep it, the GPU's skip it as they skip others.)"""
import numpy as np
import pytest

from devil_ray_amd import synthetic as syn
from test_gpu_parity import _np

pytestmark = pytest.mark.gpu


def _nets(p):
    rng = np.random.default_rng(90 + p)
    cube = syn.box_net((0.25, 0.5, 0.75), (1.25, 1.5, 1.75), p)
    cube = cube + rng.uniform(-0.02, 0.02, cube.shape)
    n, nan, inf = len(cube), np.nan, np.inf
    out = []
    for put in ([(n - 1, 2, nan)], [(n // 2, 1, inf)], [(0, 0, -inf)], [(1, 0, inf), (n - 2, 0, -inf)],
                [(k, 0, nan) for k in range(n)], [(k, c, nan) for k in range(n) for c in range(3)],
                [(k, 1, inf) for k in range(n)], [(0, c, 3e38) for c in range(3)] + [(n - 1, c, -3e38) for c in range(3)],
                [(n // 3, 0, 1e30)]):
        net = cube.copy()
        for k, c, v in put:
            net[k, c] = v
        out.append(net)
    return np.stack(out)


@pytest.mark.parametrize("p", [1, 2, 3, 4, 6])
def test_split_nonfinite_bit_exact(gpu, orc, p):
    print(f"[split nonfinite] order {p}", flush=True)
    mesh = syn.elements_from_nets(_nets(p), p)
    aabbs, prims, subrefs = gpu.UnstructuredMesh(mesh).split_elements()
    oa, op, osr = orc.split_elements(mesh)
    assert np.array_equal(_np(prims), op)
    assert np.array_equal(_np(subrefs).reshape(-1, 6).view(np.uint32), osr.view(np.uint32))
    assert np.array_equal(_np(aabbs).reshape(-1, 6).view(np.uint32), oa.view(np.uint32))
