"""Layers with a pack_layers entry: the same outputs and gradients as without one, also
where the entry holds no flipped weights."""
import pytest

from test_gpu_unet_blocks import leaf, tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flip", [True, False])
@pytest.mark.parametrize("layer", ["conv3d", "conv3d_pool", "conv3d_up"])
def test_gradients_with_an_entry_equal_those_without(gpu, layer, flip):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    if layer == "conv3d_up":
        xs, w, b, _ = tensors(gpu, [(1, 2, 4, 3), (1, 4, 8, 6)], [32, 16], 16, 8)
    else:
        xs, w, b, _ = tensors(gpu, [(1, 4, 8, 6)], [48], 16, 8)
    grads = []
    for packed in (None, sg.pack_layers([(w, flip)])[0]):
        leaves = [leaf(t) for t in (*xs, w, b)]
        y = getattr(sg, layer)(*leaves, packed=packed)
        outs = y if isinstance(y, tuple) else (y,)
        gen = torch.Generator(device=gpu).manual_seed(1)
        torch.autograd.backward(outs, [torch.randn(o.shape, generator=gen, device=gpu).to(o.dtype) for o in outs])
        grads.append([*(o.detach() for o in outs), *(t.grad for t in leaves)])
    for a, e in zip(*grads):
        assert a is not None and torch.equal(a, e)
