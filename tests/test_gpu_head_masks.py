"""head_fields takes any mask: types of more than a byte, strided and transposed views, host
arrays and the features in another layout give the fields of the contiguous bool mask."""
import numpy as np
import pytest

from test_gpu_surrogate import make_case, rand_bf16

pytestmark = pytest.mark.gpu


def forms(solid):
    import torch
    wide = torch.zeros(solid.shape[:2] + (2 * solid.shape[2],), dtype=torch.bool, device=solid.device)
    wide[..., ::2] = solid
    return {"int64": solid.long() * 256, "float": solid.float() * 0.25, "uint8": solid.to(torch.uint8) * 200,
            "int8": -solid.to(torch.int8), "strided": wide[..., ::2],
            "transposed": solid.permute(2, 1, 0).contiguous().permute(2, 1, 0), "array": solid.cpu().numpy(),
            "float array": solid.cpu().numpy().astype(np.float64)}


@pytest.mark.parametrize("form", ["int64", "float", "uint8", "int8", "strided", "transposed", "array", "float array"])
def test_any_mask_gives_the_same_fields(gpu, form):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    x = rand_bf16((6, 5, 9, 16), 90).to(gpu)
    _, wt, b = make_case((1, 1, 1, 1, 16, 16, 1), 91)
    wt, b = wt.to(gpu), b.to(gpu)
    solid = (torch.rand((4, 5, 7), generator=torch.Generator().manual_seed(92)) < 0.4).to(gpu)
    want = sg.head_fields(x, wt, b, solid, (1, 0, 2), 2.0, 3.0, False)
    got = sg.head_fields(x, wt, b, forms(solid)[form], (1, 0, 2), 2.0, 3.0, False)
    turned = x.permute(1, 0, 2, 3).contiguous().permute(1, 0, 2, 3)
    view = sg.head_fields(turned, wt, b, solid, (1, 0, 2), 2.0, 3.0, False)
    for g, v, e in zip(got, view, want):
        assert torch.equal(g, e) and torch.equal(v, e)
