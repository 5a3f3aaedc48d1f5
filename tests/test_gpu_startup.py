"""Compaction over the list order's divisions and the scan's rounds against numpy, and
the padding that initialisation clears."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def list_order(shape, band):
    """Dense indices in list order: bands of rows j, plane after plane in a band."""
    idx = np.arange(np.prod(shape)).reshape(shape)
    band = band if 0 < band < shape[1] else shape[1]
    return np.concatenate([idx[:, j:j + band].reshape(-1) for j in range(0, shape[1], band)])


# one and several rounds of the scan (8,192 tiles of 1,024 nodes), last bands of 1 and R - 1 rows, prime extents
@pytest.mark.parametrize("shape,band", [((1, 1, 1), 32), ((3, 33, 7), 32), ((5, 63, 31), 32), ((11, 13, 17), 4),
                                        ((7, 8, 129), 1), ((17, 70, 9), 0), ((210, 200, 200), 32), ((97, 301, 293), 7)])
def test_fluid_list_equals_numpy(gpu, shape, band):
    import torch
    from taichi_lbm3d_amd import LB3D_Solver_Single_Phase
    rng = np.random.default_rng(sum(shape))
    solid = (rng.random(shape) < 0.6).astype(np.int8)
    solid.reshape(-1)[-1] = 0
    s = LB3D_Solver_Single_Phase(*shape, sparse_storage=True)
    s.band_rows = band
    s.solid.from_numpy(solid)
    s.init_simulation()
    order = list_order(shape, band)
    want = order[solid.reshape(-1)[order] == 0]
    assert s.n_fluid == len(want)
    np.testing.assert_array_equal(s._dev["cells"][:s.n_fluid].cpu().numpy(), want)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("cells", [1, 63, 64, 65, 257])
def test_init_clears_the_padding(gpu, dtype, cells):
    import torch
    from taichi_lbm3d_amd import LB3D_Solver_Single_Phase, _lib
    s = LB3D_Solver_Single_Phase(1, 1, cells + 1, sparse_storage=True, dtype=dtype)
    solid = np.zeros((1, 1, cells + 1), np.int8)
    solid[0, 0, 0] = 1
    s.solid.from_numpy(solid)
    s.init_simulation()
    stride = _lib.lib().size("lbm3d_slot_stride", cells)
    g = s._dev["g"].view(19, stride)
    g.fill_(7.0)
    s._init_state()
    assert (g[:, cells:] == 0).all()
    assert (g[:, :cells] != 7.0).all()
