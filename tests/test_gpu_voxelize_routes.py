"""lbm3d_voxelize_blocks on every route it takes: the same flags as lbm3d_voxelize, node by
node, for few and large triangles, many, meshes that leave most nodes open, and times
of the same order where most blocks stay open."""
import numpy as np
import pytest

from test_gpu_voxelize import both

pytestmark = pytest.mark.gpu


def boxes(count, n, seed=5):
    from taichi_lbm3d_amd.stl import box_mesh
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        c, r = rng.uniform(.25, .75, 3) * n, rng.uniform(.08, .22) * n
        out.append(box_mesh(c - r, c + r))
    return np.concatenate(out)


def soup(count, n, size, seed=7):
    rng = np.random.default_rng(seed)
    return rng.uniform(0, n, (count, 1, 3)) + rng.uniform(-size, size, (count, 3, 3))


# triangles and grids on both sides of the rules: under 9e6 nodes x triangles (or 106
# triangles on a small grid) every node is summed at once; up to 566 triangles the share of
# open blocks decides on the device
@pytest.mark.parametrize("count", [1, 8, 9, 16, 47, 48])
@pytest.mark.parametrize("n", [31, 49, 72])
def test_overlapping_boxes(gpu, count, n):
    want, got = both(gpu, boxes(count, n), (0.0, 0.0, 0.0), 1.0, (n, n - 3, n + 2))
    assert 0 < want.sum() < want.size
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("count,n,size", [(106, 30, 4.0), (105, 30, 4.0), (300, 50, 8.0), (600, 41, 5.0),
                                          (3000, 30, 2.0)])
def test_triangle_soups(gpu, count, n, size):
    want, got = both(gpu, soup(count, n, size), (0.0, 0.0, 0.0), 1.0, (n, n, n + 1))
    np.testing.assert_array_equal(got, want)


# a corner that is no number leaves every node open: 1, 4 and 8 of them a wave, the last
# wave's group not full
@pytest.mark.parametrize("shape", [(11, 9, 10), (30, 31, 29), (47, 46, 45)])
@pytest.mark.parametrize("count", [601, 640])
def test_every_node_open(gpu, shape, count):
    tris = soup(count, 30, 3.0)
    tris[17, 2, 1] = np.nan
    want, got = both(gpu, tris, (0.0, 0.0, 0.0), 1.0, shape)
    np.testing.assert_array_equal(got, want)


# more than 65,536 triangles: a closed surface goes block by block, a soup and a mesh
# without numbers go to the plain kernel
@pytest.mark.parametrize("kind", ["closed", "soup", "not a number"])
@pytest.mark.parametrize("shape", [(1, 1, 2), (10, 9, 11)])
def test_large_meshes(gpu, kind, shape):
    from taichi_lbm3d_amd.stl import sphere_mesh
    if kind == "closed":
        tris = sphere_mesh((5.2, 4.1, 4.9), 3.7, 6)
    else:
        tris = soup(66000, 10, 1.0)
        if kind == "not a number":
            tris[0, 0, 0] = np.nan
    want, got = both(gpu, tris, (0.0, 0.0, 0.0), 1.0, shape)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("mesh", ["16 boxes", "48 boxes"])
def test_surfaces_everywhere_cost_no_more_than_the_plain_kernel_twice(gpu, mesh):
    """Where blocks decide little the call falls back in time: 16 and 48 overlapping boxes on
    96 x 96 x 96 nodes (0.9 and 2.5 ms by the plain kernel, 14 and 20 ms with the counters and
    FP64 sums of every open node)."""
    import torch
    from taichi_lbm3d_amd import _lib
    lib = _lib.lib()
    shape = (96, 96, 96)
    t = torch.from_numpy(np.ascontiguousarray(boxes(int(mesh.split()[0]), 96), np.float32)).to(gpu)
    out = torch.empty(shape, dtype=torch.int8, device=gpu)
    size = lib.size("lbm3d_voxelize_workspace_bytes", *shape)
    ws = torch.empty(size, dtype=torch.uint8, device=gpu)
    args = (torch.cuda.current_stream().cuda_stream, t.data_ptr(), len(t), 0.0, 0.0, 0.0, 1.0, *shape, out.data_ptr())

    def best(name, *more):
        times = []
        for _ in range(6):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            lib.call(name, *args, *more)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    assert best("lbm3d_voxelize_blocks", ws.data_ptr(), size) < 2 * best("lbm3d_voxelize")
