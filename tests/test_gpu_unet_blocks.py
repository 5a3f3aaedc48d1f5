"""The surrogate's fused blocks -- convolution with pooling, convolution of an
upsampled and a skip part -- against the plain layers and PyTorch operations
they replace: outputs and gradients bit for bit, except the upsampling's
gradient (8 BF16 terms summed in FP32, whose order is not torch's)."""
import pytest

pytestmark = pytest.mark.gpu


def tensors(gpu, shape, cins, cout, seed):
    import torch
    gen = torch.Generator(device=gpu).manual_seed(seed)
    xs = [torch.randn(tuple(s) + (c,), generator=gen, device=gpu).to(torch.bfloat16) for s, c in zip(shape, cins)]
    k = 27 * sum(cins)
    w = torch.zeros((cout, (k + 31) // 32 * 32), device=gpu)
    w[:, :k] = torch.randn((cout, k), generator=gen, device=gpu) / k ** 0.5
    b = torch.randn(cout, generator=gen, device=gpu) * 0.1
    return xs, w, b, gen


def pool(x):
    n, d, h, w, c = x.shape
    return x.view(n, d // 2, 2, h // 2, 2, w // 2, 2, c).amax(dim=(2, 4, 6))


def up(x):
    n, d, h, w, c = x.shape
    return x[:, :, None, :, None, :, None, :].expand(n, d, 2, h, 2, w, 2, c).reshape(n, 2 * d, 2 * h, 2 * w, c)


def leaf(t):
    return t.clone().requires_grad_(True)


# n, d, h, w, cin, cout: remainders of the columns and bricks, several runs of
# planes, every kernel that pools
POOLED = [(1, 2, 2, 2, 16, 16), (2, 6, 18, 34, 16, 16), (1, 70, 16, 16, 16, 16), (1, 4, 10, 18, 16, 32),
          (1, 4, 8, 14, 16, 64), (2, 6, 10, 18, 32, 32), (1, 4, 6, 20, 32, 16), (1, 6, 12, 16, 48, 32),
          (1, 4, 10, 18, 64, 64), (2, 4, 6, 10, 80, 32), (1, 4, 10, 6, 64, 128), (1, 6, 10, 18, 128, 16)]


@pytest.mark.parametrize("form", POOLED)
@pytest.mark.parametrize("periodic", [False, True])
def test_pooled_convolution_forward(gpu, form, periodic):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout = form
    (x,), wt, b, _ = tensors(gpu, [(n, d, h, w)], [cin], cout, 1)
    with torch.no_grad():
        y, p = sg.conv3d_pool(x, wt, b, periodic)
        ref = sg.conv3d(x, wt, b, 3, True, periodic=periodic)
    assert torch.equal(y, ref)
    assert torch.equal(p, pool(ref))


@pytest.mark.parametrize("form", POOLED)
def test_pooled_convolution_gradients(gpu, form):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout = form
    (x,), wt, b, gen = tensors(gpu, [(n, d, h, w)], [cin], cout, 2)
    b = b - 0.5  # blocks whose maximum is 0 in all 8 voxels
    gy = torch.randn((n, d, h, w, cout), generator=gen, device=gpu).to(torch.bfloat16)
    gp = torch.randn((n, d // 2, h // 2, w // 2, cout), generator=gen, device=gpu).to(torch.bfloat16)
    got, want = [leaf(t) for t in (x, wt, b)], [leaf(t) for t in (x, wt, b)]
    y, p = sg.conv3d_pool(*got)
    torch.autograd.backward([y, p], [gy, gp])
    r = sg.conv3d(*want, 3, True)
    torch.autograd.backward([r, pool(r)], [gy, gp])
    for name, a, e in zip(("dx", "dw", "db"), got, want):
        assert torch.equal(a.grad, e.grad), name


# n, d, h, w (full extents), c_low, c_skip, cout
UP = [(1, 2, 2, 2, 16, 16, 16), (2, 6, 18, 34, 32, 16, 16), (1, 4, 10, 18, 16, 16, 32), (1, 8, 8, 16, 16, 32, 32),
      (1, 4, 10, 18, 64, 32, 32), (2, 4, 6, 10, 128, 64, 64), (1, 34, 40, 36, 128, 64, 64), (1, 2, 4, 6, 64, 16, 16),
      (1, 70, 16, 16, 32, 16, 16)]


@pytest.mark.parametrize("form", UP)
@pytest.mark.parametrize("periodic", [False, True])
def test_upsampled_convolution_forward(gpu, form, periodic):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cl, cs, cout = form
    (low, skip), wt, b, _ = tensors(gpu, [(n, d // 2, h // 2, w // 2), (n, d, h, w)], [cl, cs], cout, 3)
    with torch.no_grad():
        y = sg.conv3d_up(low, skip, wt, b, periodic)
        ref = sg.conv3d(torch.cat([up(low), skip], -1), wt, b, 3, True, periodic=periodic)
    assert torch.equal(y, ref)


@pytest.mark.parametrize("form", UP)
def test_upsampled_convolution_gradients(gpu, form):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cl, cs, cout = form
    (low, skip), wt, b, gen = tensors(gpu, [(n, d // 2, h // 2, w // 2), (n, d, h, w)], [cl, cs], cout, 4)
    gy = torch.randn((n, d, h, w, cout), generator=gen, device=gpu).to(torch.bfloat16)
    got, want = [leaf(t) for t in (low, skip, wt, b)], [leaf(t) for t in (low, skip, wt, b)]
    sg.conv3d_up(*got).backward(gy)
    sg.conv3d(torch.cat([up(want[0]), want[1]], -1), want[2], want[3], 3, True).backward(gy)
    for name, a, e in zip(("skip", "w", "b"), got[1:], want[1:]):
        assert torch.equal(a.grad, e.grad), name
    # both round an FP32 sum of the same 8 values to BF16: at most one place apart
    a, e = got[0].grad.float(), want[0].grad.float()
    assert ((a - e).abs() <= 2 ** -7 * e.abs() + 1e-6 * e.abs().max()).all()
    assert (a != e).float().mean() < 1e-2


@pytest.mark.parametrize("form", [(1, 6, 10, 18, 16, 32, 48), (1, 12, 20, 34, 32, 32, 48), (2, 4, 8, 16, 48, 16, 96)])
def test_data_gradient_sums_blocks(gpu, form):
    """The C call at channel counts that autograd does not reach: the parts are the plain
    data gradient's, the low one summed over blocks of 8 exactly representable values."""
    import torch
    from taichi_lbm3d_amd import _lib
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cl, cs, cout = form
    gen = torch.Generator(device=gpu).manual_seed(6)
    # small whole numbers: every output is a whole number below 2^8 with few terms, so BF16 holds it
    g = torch.randint(0, 2, (n, d, h, w, cout), generator=gen, device=gpu).to(torch.bfloat16)
    wt = (torch.rand((cout, 27 * (cl + cs)), generator=gen, device=gpu) < 0.02).float()
    wt = torch.nn.functional.pad(wt, (0, _lib.lib().cdll.lbm3d_conv_kpad(cl + cs, 3) - wt.shape[1]))
    _, flipped = sg.pack_weights(wt, True)
    full = sg.conv_fwd_packed(g, flipped, None, cl + cs, False)
    d_low = torch.empty((n, d // 2, h // 2, w // 2, cl), dtype=torch.bfloat16, device=gpu)
    d_skip = torch.empty((n, d, h, w, cs), dtype=torch.bfloat16, device=gpu)
    _lib.lib().call("lbm3d_conv3d_dgrad_up", torch.cuda.current_stream().cuda_stream, g.data_ptr(), flipped.data_ptr(),
                    d_low.data_ptr(), d_skip.data_ptr(), n, d, h, w, cl, cs, cout)
    assert torch.equal(d_skip, full[..., cl:])
    blocks = full[..., :cl].float().reshape(n, d // 2, 2, h // 2, 2, w // 2, 2, cl).sum((2, 4, 6))
    assert torch.equal(d_low, blocks.to(torch.bfloat16))  # sums of whole numbers are exact before the rounding


def test_odd_extents_and_missing_relu_are_refused(gpu):
    import torch
    from taichi_lbm3d_amd import _lib
    from taichi_lbm3d_amd import surrogate as sg
    (x,), wt, b, _ = tensors(gpu, [(1, 3, 4, 4)], [16], 16, 5)
    with pytest.raises(_lib.LbmError, match="even"):
        sg.conv3d_pool(x, wt, b)
    (low, skip), wt, b, _ = tensors(gpu, [(1, 2, 2, 2), (1, 4, 4, 5)], [16, 16], 16, 5)
    with pytest.raises(_lib.LbmError, match="even"):
        sg.conv3d_up(low, skip, wt, b)
