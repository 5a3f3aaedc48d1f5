"""lbm3d_voxelize_blocks against lbm3d_voxelize, node by node: the same flags for
closed, open, nested and reversed meshes, triangle soups, surfaces through the
nodes, and coordinates far from or tiny beside the cell size."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def both(gpu, tris, origin, dx, shape):
    import torch
    from taichi_lbm3d_amd import _lib
    lib = _lib.lib()
    tris = np.ascontiguousarray(np.asarray(tris, np.float32).reshape(-1, 9))
    t = torch.from_numpy(tris if len(tris) else np.zeros((1, 9), np.float32)).to(gpu)
    out = [torch.full(shape, 7, dtype=torch.int8, device=gpu) for _ in range(2)]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    args = (stream, ctypes.c_void_p(t.data_ptr()), len(tris), *map(float, origin), float(dx), *shape)
    lib.call("lbm3d_voxelize", *args, ctypes.c_void_p(out[0].data_ptr()))
    size = lib.size("lbm3d_voxelize_workspace_bytes", *shape)
    ws = torch.empty(size, dtype=torch.uint8, device=gpu)
    lib.call("lbm3d_voxelize_blocks", *args, ctypes.c_void_p(out[1].data_ptr()), ctypes.c_void_p(ws.data_ptr()), size)
    return out[0].cpu().numpy(), out[1].cpu().numpy()


def meshes():
    from taichi_lbm3d_amd.stl import box_mesh, sphere_mesh
    rng = np.random.default_rng(3)
    ball = sphere_mesh((11.3, 9.6, 10.1), 7.2, 3)
    small = sphere_mesh((11.3, 9.6, 10.1), 3.1, 2)
    box = box_mesh((3.0, 4.0, 2.0), (15.0, 12.0, 18.0))  # faces, edges and corners on nodes
    two = box_mesh((15.0, 4.0, 2.0), (19.0, 12.0, 18.0))
    return {
        "empty": np.zeros((0, 3, 3)),
        "one": ball[:1],
        "sphere": ball,
        "shell": np.concatenate([ball, small[:, ::-1]]),
        "doubled": np.concatenate([ball, ball, small]),
        "inside out": ball[:, ::-1],
        "open": ball[ball.mean(1)[:, 2] < 12.0],
        "box on nodes": box,
        "boxes sharing a face": np.concatenate([box, two]),
        "soup": rng.uniform(0, 22, (150, 3, 3)),
        "slivers": np.concatenate([ball, np.repeat(rng.uniform(5, 15, (20, 1, 3)), 3, 1),
                                   rng.uniform(5, 15, (20, 1, 3)) + np.linspace(0, 1, 3)[None, :, None]]),
        "far corner": np.concatenate([ball, [[[1e9, 0, 0], [0, 1e9, 0], [0, 0, 1e9]]]]),
        "huge": np.concatenate([ball, [[[1e30, 0, 0], [0, 1e30, 0], [0, 0, 1e30]]]]),
        "not a number": np.concatenate([ball, [[[np.nan, 0, 0], [0, 1, 0], [0, 0, 1]]]]),
    }


NAMES = ["empty", "one", "sphere", "shell", "doubled", "inside out", "open", "box on nodes", "boxes sharing a face",
         "soup", "slivers", "far corner", "huge", "not a number"]


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("shape", [(1, 1, 1), (23, 21, 22), (8, 16, 33)])
def test_blocks_give_every_nodes_flag(gpu, name, shape):
    want, got = both(gpu, meshes()[name], (0.0, 0.0, 0.0), 1.0, shape)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("scale, origin", [(1e-6, (0, 0, 0)), (1e-13, (0, 0, 0)), (1.0, (1e6, -1e6, 3e5)),
                                           (250.0, (-1e4, 0, 1e3)), (0.3, (0.1, 0.2, 0.3))])
@pytest.mark.parametrize("name", ["sphere", "open", "box on nodes"])
def test_any_scale_and_origin(gpu, name, scale, origin):
    tris = meshes()[name] * scale + np.array(origin)
    want, got = both(gpu, tris, origin, scale, (23, 21, 22))
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("radius,level,dx", [(60.0, 3, 1.0), (60.0, 4, 1.0), (4.0, 4, 0.05), (200.0, 2, 7.0)])
def test_near_and_far_triangles_give_the_same_flags(gpu, radius, level, dx):
    """A surface of many triangles, most of them far from any block, some blocks with more
    near ones than a wave has lanes; triangles smaller and larger than a cell."""
    from taichi_lbm3d_amd.stl import sphere_mesh
    shape = (26, 19, 33)
    origin = np.array([radius * 0.8, -9 * dx, 3 * dx])
    ball = sphere_mesh((0.0, 0.0, 0.0), radius, level)
    inner = sphere_mesh((radius, 0.0, 8 * dx), 6 * dx, 2)
    ref, got = both(gpu, np.concatenate([ball, inner]), origin, dx, shape)
    assert 0 < ref.sum() < ref.size
    np.testing.assert_array_equal(got, ref)
