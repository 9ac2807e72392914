"""The scan of a sort's digit counts on both sides of the count up to which one block takes it (10,240 counts, 40 tiles of 4,096
keys), at a tile's edges and at the smallest sizes: points located in Morton order get the records that they get in theirs."""
import pytest
import torch

from devil_ray_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 4095, 4096, 4097, 32 * 4096, 40 * 4096 - 1, 40 * 4096, 40 * 4096 + 1, 41 * 4096 + 5, 128 * 4096])
def test_morton_order_keeps_every_point(gpu, n):
    print(f"[sort scan] {n} points", flush=True)
    mesh = gpu.UnstructuredMesh(syn.hex_mesh(4, 2, 0.05, 0.01, 3))
    g = torch.Generator("cuda").manual_seed(n)
    pts = torch.rand((n, 3), device="cuda", generator=g).reshape(-1)
    plain = mesh.locate(pts, gpu.LocateOptions(launch=1))
    assert torch.equal(mesh.locate(pts, gpu.LocateOptions(launch=1, coherent_order=True)), plain)
    assert int((plain.view(torch.int32).reshape(-1, 4)[:, 0] >= 0).sum()) >= n // 2
