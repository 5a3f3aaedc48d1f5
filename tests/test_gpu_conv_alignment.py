"""Operands that do not start on 16 bytes, or are no contiguous tensors, give the results of
their copies; the C calls, which cannot copy, refuse them."""
import pytest

from test_gpu_unet_blocks import leaf, tensors

pytestmark = pytest.mark.gpu


def moved(t, by):
    """The same values, `by` elements after an aligned address."""
    import torch
    flat = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)[by:]
    flat.copy_(t.reshape(-1))
    return flat.view(t.shape)


@pytest.mark.parametrize("by", [1, 2, 4])
@pytest.mark.parametrize("layer", ["conv3d", "conv1", "conv3d_pool", "conv3d_up", "conv_head"])
def test_any_start_gives_the_same_results(gpu, layer, by):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    if layer == "conv3d_up":
        xs, w, b, _ = tensors(gpu, [(1, 2, 4, 9), (1, 4, 8, 18)], [16, 32], 16, 9)
    else:
        xs, w, b, _ = tensors(gpu, [(2, 4, 8, 18)], [16], 16, 9)
    if layer in ("conv1", "conv_head"):
        w = w[:, :32].contiguous()
        w[:, 16:] = 0

    def call(*t):
        if layer == "conv1":
            return sg.conv3d(*t, 1, True)
        return getattr(sg, layer)(*t)

    results = []
    for shift in (0, by):
        leaves = [leaf(t) for t in (*xs, w, b)]
        y = call(*(moved(t, shift) if shift else t for t in leaves))
        outs = y if isinstance(y, tuple) else (y,)
        gen = torch.Generator(device=gpu).manual_seed(1)
        gys = [torch.randn(o.shape, generator=gen, device=gpu).to(o.dtype) for o in outs]
        torch.autograd.backward(outs, [moved(g, shift) if shift else g for g in gys])
        results.append([*(o.detach() for o in outs), *(t.grad for t in leaves)])
    for a, e in zip(*results):
        assert torch.equal(a, e)


def test_helpers_take_views(gpu):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    (x,), w, b, gen = tensors(gpu, [(1, 3, 5, 17)], [32], 16, 10)
    dy = torch.randn((1, 3, 5, 17, 16), generator=gen, device=gpu).to(torch.bfloat16)
    wb = w.to(torch.bfloat16)
    turned = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)
    for f in (turned, lambda t: moved(t, 3)):
        assert torch.equal(sg.conv_fwd(f(x), moved(wb, 1), b, 16, 3, True), sg.conv_fwd(x, wb, b, 16, 3, True))
        assert torch.equal(sg.conv_wgrad(f(x), f(dy), 3), sg.conv_wgrad(x, dy, 3))
        assert torch.equal(sg.conv_dgrad(f(dy), wb, 32, 3), sg.conv_dgrad(dy, wb, 32, 3))


def test_c_calls_refuse_other_starts(gpu):
    import torch
    from taichi_lbm3d_amd import _lib
    from taichi_lbm3d_amd import surrogate as sg
    (low, x), w, b, _ = tensors(gpu, [(1, 2, 2, 2), (1, 4, 4, 4)], [16, 16], 16, 11)
    w32 = torch.zeros((16, 864), device=gpu)
    y, off = torch.empty_like(x), moved(x, 1)
    wp, wt = sg.pack_weights(w, True)
    wu, wut = sg.pack_weights(w32, True)
    s, dims = torch.cuda.current_stream().cuda_stream, (1, 4, 4, 4)
    dw, ws = torch.empty_like(w), torch.empty(1 << 22, dtype=torch.uint8, device=gpu)
    p = lambda t: t.data_ptr()
    for name, args in (
            ("lbm3d_conv3d_fwd", (p(off), p(w.to(torch.bfloat16)), None, p(y), *dims, 16, 16, 3, 0)),
            ("lbm3d_conv3d_fwd_packed", (p(off), p(wp), None, p(y), *dims, 16, 16, 0)),
            ("lbm3d_conv3d_fwd_pool", (p(off), p(wp), None, p(y), p(low), *dims, 16, 16, 1)),
            ("lbm3d_conv3d_fwd_up", (p(moved(low, 1)), p(x), p(wu), None, p(y), *dims, 16, 16, 16, 0)),
            ("lbm3d_conv3d_dgrad_up", (p(off), p(wut), p(low), p(y), *dims, 16, 16, 16)),
            ("lbm3d_conv3d_wgrad", (p(x), p(off), p(dw), *dims, 16, 16, 3, p(ws), ws.numel()))):
        with pytest.raises(_lib.LbmError, match="16 bytes"):
            _lib.lib().call(name, s, *args)
