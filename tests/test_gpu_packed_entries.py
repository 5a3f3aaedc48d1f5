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


# both sides of the rule that reads weights of other types as rows, with and without gradients
@pytest.mark.parametrize("cin, cout", [(16, 16), (48, 32), (48, 64), (64, 16), (128, 128)])
@pytest.mark.parametrize("kind", ["bfloat16", "float64"])
def test_weights_of_other_types_give_the_rounded_weights_results(gpu, cin, cout, kind):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    (x,), w, b, gen = tensors(gpu, [(1, 5, 9, 17)], [cin], cout, 12)
    gy = torch.randn((1, 5, 9, 17, cout), generator=gen, device=gpu).to(torch.bfloat16)
    w = w.to(torch.bfloat16)
    results = []
    for wk in (w.float(), w.to(getattr(torch, kind))):
        leaves = [leaf(t) for t in (x, wk, b)]
        with torch.no_grad():
            y0 = sg.conv3d(*leaves, 3, True, periodic=True)
        y = sg.conv3d(*leaves, 3, True)
        y.backward(gy)
        results.append([y0, y.detach(), *(t.grad for t in leaves)])
    for a, e in zip(*results):  # the weights' gradient comes in their type
        assert torch.equal(a.to(e.dtype), e)


def test_bf16_weights_pack_as_their_floats(gpu):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    _, w, _, _ = tensors(gpu, [(1, 1, 1, 1)], [48], 32, 13)
    wb = w.to(torch.bfloat16)
    for a, e in zip(sg.pack_weights(wb, True), sg.pack_weights(wb.float(), True)):
        assert torch.equal(a, e)
