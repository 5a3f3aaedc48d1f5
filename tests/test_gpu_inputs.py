"""The surrogate's inputs from the geometry: mask and periodic distance, FP32
pairs and the network's 16-channel BF16 form, against a brute-force nearest
solid cell under minimum-image wrap (valid for extents below the margin too,
where the padded EDT of the oracle is not)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# extents below, at and above the margin; one-voxel axes; a last wave that is not full
SHAPES = [(1, 1, 1), (1, 7, 65), (3, 2, 64), (24, 25, 23), (49, 5, 50), (31, 33, 63)]


def nearest_solid(solid, margin):
    cells = np.indices(solid.shape).reshape(3, -1)
    best = np.full(cells.shape[1], float(margin) ** 2)
    for p in np.argwhere(solid):
        off = np.abs(cells - p[:, None])
        off = np.minimum(off, np.array(solid.shape)[:, None] - off)
        best = np.minimum(best, (off.astype(np.float64) ** 2).sum(0))
    return np.sqrt(best).reshape(solid.shape).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("fraction", [0.0, 0.01, 0.1])
@pytest.mark.parametrize("margin", [1, 2, 7, 24, 63, 64])
def test_distance_equals_edt_for_every_margin(gpu, shape, fraction, margin):
    import torch
    from taichi_lbm3d_amd.surrogate import periodic_distance
    rng = np.random.default_rng(sum(shape) + int(100 * fraction))
    solid = (rng.random(shape) < fraction).astype(np.uint8)
    got = periodic_distance(torch.from_numpy(solid).to(gpu), margin=margin).cpu().numpy()
    np.testing.assert_array_equal(got, nearest_solid(solid, margin))


@pytest.mark.parametrize("dtype", ["uint8", "int8", "bool", "float32", "int64"])
def test_inputs_are_mask_and_scaled_distance(gpu, dtype):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    rng = np.random.default_rng(5)
    solid = rng.random((2, 11, 13, 17)) < 0.1
    t = torch.from_numpy(solid).to(gpu).to(getattr(torch, dtype))
    if dtype == "int8":
        t = -t  # negative values are solid too
    dist = sg.periodic_distance(t)
    pair = sg.make_inputs(t)
    want = torch.stack([torch.from_numpy(solid).to(gpu).float(), dist / sg.DIST_SCALE], dim=-1)
    assert torch.equal(pair, want)
    assert torch.equal(sg.network_inputs(t), sg.to_network_input(want))
    assert torch.equal(sg.make_inputs(t.transpose(1, 3)), sg.make_inputs(t.transpose(1, 3).contiguous()))


@pytest.mark.parametrize("shape", [(257, 3, 5), (3, 257, 5), (256, 2, 70), (2, 256, 64), (33, 16, 129)])
@pytest.mark.parametrize("margin", [3, 24, 63])
def test_lines_at_the_limit_of_the_lds(gpu, shape, margin):
    """Lines of 256 and 257 voxels along the outer and the middle axis, batched; whole and partial waves."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    rng = np.random.default_rng(margin)
    solids = [(rng.random(shape) < f).astype(np.uint8) for f in (0.004, 0.03)]
    batch = torch.from_numpy(np.stack(solids)).to(gpu)
    want = np.stack([nearest_solid(s, margin) for s in solids])
    np.testing.assert_array_equal(sg.periodic_distance(batch, margin=margin).cpu().numpy(), want)
    if margin == 24:
        pair = torch.stack([batch.float(), torch.from_numpy(want).to(gpu) / sg.DIST_SCALE], dim=-1)
        assert torch.equal(sg.network_inputs(batch), sg.to_network_input(pair))
