"""Odd steps that find their cells' places through the tile descriptors against the
cell-list lookup, where a wave's words can go wrong: words without a fluid cell, a
wave that starts inside a word, waves of one and of 64 words, rows of one cell, of a
word's edge and of many words, a last block that is not full, blocks over two
segments of the list."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# extents, fluid fraction, rows per band
GRIDS = [((9, 40, 1), 0.7, 32), ((7, 50, 31), 0.02, 32), ((7, 50, 32), 0.5, 8), ((5, 37, 33), 1.0, 32),
         ((6, 40, 64), 0.03, 16), ((8, 33, 65), 0.9, 32), ((4, 12, 300), 0.1, 5), ((3, 8, 700), 0.6, 32),
         ((1, 1, 257), 1.0, 32), ((2, 3, 2047), 0.3, 1), ((20, 64, 48), 0.35, 0)]


@pytest.mark.parametrize("shape,fraction,band", GRIDS)
@pytest.mark.parametrize("dtype", ["f32", "bf16sr"])
def test_places_from_descriptors_equal_the_cell_list(gpu, shape, fraction, band, dtype):
    import torch
    from taichi_lbm3d_amd import LB3D_Solver_Single_Phase
    rng = np.random.default_rng(sum(shape))
    solid = (rng.random(shape) >= fraction).astype(np.int8)
    solid[0, 0, 0] = 0
    out = []
    for tiles in (False, True):
        s = LB3D_Solver_Single_Phase(*shape, sparse_storage=True, dtype=dtype)
        s.use_tiles, s.band_rows = tiles, band
        s.solid.from_numpy(solid)
        s.set_viscosity(0.3)
        s.set_force([1e-4, -2e-4, 3e-4])
        s.init_simulation()
        s.run(6)
        torch.cuda.synchronize()
        out.append(s._dev["g"].cpu())
    assert torch.isfinite(out[0].float()).all() and out[0].float().abs().max() > 0
    assert torch.equal(out[0], out[1])
