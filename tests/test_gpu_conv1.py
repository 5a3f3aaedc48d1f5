"""1x1x1 convolutions of 1, 2 and 4 interleaved channel tiles and their weight gradients
against FP64 products of the same bf16 operands, and the wide ones' time against their bytes."""
import pytest

pytestmark = pytest.mark.gpu


def layer(gpu, voxels, cin, cout, seed):
    import torch
    gen = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn((1, 1, 1, voxels, cin), generator=gen, device=gpu).to(torch.bfloat16)
    w = torch.zeros((cout, (cin + 31) // 32 * 32), device=gpu)
    w[:, :cin] = torch.randn((cout, cin), generator=gen, device=gpu) / cin ** 0.5
    b = torch.randn(cout, generator=gen, device=gpu)
    dy = torch.randn((1, 1, 1, voxels, cout), generator=gen, device=gpu).to(torch.bfloat16)
    return x, w.to(torch.bfloat16), b, dy


@pytest.mark.parametrize("cin, cout", [(16, 16), (48, 32), (16, 48), (80, 64), (32, 96), (16, 128), (240, 240),
                                       (256, 256)])
@pytest.mark.parametrize("voxels", [1, 17, 255, 1031])
@pytest.mark.parametrize("relu", [False, True])
def test_forward(gpu, voxels, cin, cout, relu):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    x, w, b, _ = layer(gpu, voxels, cin, cout, 1)
    exact = x.double().view(-1, cin) @ w[:, :cin].double().t()
    for bias in (b, None):
        y = sg.conv_fwd(x, w, bias, cout, 1, relu).double().view(-1, cout)
        want = exact + (bias.double() if bias is not None else 0.0)
        want = want.relu() if relu else want
        # at most 258 FP32 additions of terms whose sizes sum to at most 4 sqrt(cin), then half a bf16 place (8 bits)
        assert ((y - want).abs() <= 2 ** -8 * want.abs() * 1.01 + 258 * 2 ** -24 * 4 * cin ** 0.5).all()


@pytest.mark.parametrize("cin, cout", [(16, 16), (32, 16), (16, 32), (48, 64), (128, 96), (240, 240)])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 5, 9, 33), (1, 40, 33, 50)])
def test_weight_gradient(gpu, shape, cin, cout):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    gen = torch.Generator(device=gpu).manual_seed(2)
    x = torch.randn(shape + (cin,), generator=gen, device=gpu).to(torch.bfloat16)
    dy = torch.randn(shape + (cout,), generator=gen, device=gpu).to(torch.bfloat16)
    dw = sg.conv_wgrad(x, dy, 1).double()
    want = dy.double().view(-1, cout).t() @ x.double().view(-1, cin)
    size = dy.double().abs().view(-1, cout).t() @ x.double().abs().view(-1, cin)
    # sums of 32 in an MFMA, of at most 16 of those in a wave, then of the sets 16 at a time: fewer than 200 roundings
    assert ((dw[:, :cin] - want).abs() <= 200 * 2 ** -24 * size).all()
    assert (dw[:, cin:] == 0).all()


def test_wide_outputs_cost_their_bytes(gpu):
    """16 -> 128 channels at 2 x 96^3 and 32 -> 32 weights' gradients at 2 x 128^3 against a copy
    of their largest tensors (168 and 139 us against about 180 and 110; 337 and 338 with narrow
    stores and with every tile's voxels read anew)."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg

    def best(f):
        times = []
        for _ in range(8):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            f()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    x, w, b, dy = layer(gpu, 2 * 96 ** 3, 16, 128, 3)
    assert best(lambda: sg.conv_fwd(x, w, b, 128, 1, True)) < 1.5 * best(lambda: torch.empty_like(dy).copy_(dy))
    x, _, _, dy = layer(gpu, 2 * 128 ** 3, 32, 32, 4)
    x, dy = (t.view(2, 128, 128, 128, 32) for t in (x, dy))
    assert best(lambda: sg.conv_wgrad(x, dy, 1)) < 2 * best(lambda: torch.empty_like(dy).copy_(dy))
