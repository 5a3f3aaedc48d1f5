"""The brick convolutions at the sizes where a workgroup takes 2 or 4 channel tiles or loops
over several bricks: plain against FP32 CPU convolutions, pooled, upsampled and split ones
against the plain kernel of the same operands, bit for bit.

A workgroup takes 4 tiles of 16 output channels (2 where 4 do not divide them) if that leaves
512 workgroups over the bricks of 2 x 8 x 16 voxels."""
import pytest

from test_gpu_surrogate import cpu_conv, make_case
from test_gpu_unet_blocks import pool, tensors, up

pytestmark = pytest.mark.gpu


def tiles_of(n, d, h, w, cout):
    """(channel tiles of a workgroup, bricks)"""
    bricks, tiles = n * -(-d // 2) * -(-h // 8) * -(-w // 16), cout // 16
    ct = 4 if tiles % 4 == 0 else 2 if tiles % 2 == 0 else 1
    while ct > 1 and bricks * (tiles // ct) < 512:
        ct //= 2
    return ct, bricks


# n, d, h, w, cin, cout, channel tiles; the last two loop over bricks with an odd number of 16-channel chunks
PLAIN = [(2, 33, 45, 50, 64, 64, 4), (1, 33, 41, 49, 64, 128, 4), (2, 33, 45, 50, 64, 32, 2),
         (1, 31, 43, 50, 64, 96, 2), (2, 33, 60, 50, 80, 16, 1), (2, 33, 60, 50, 112, 32, 2)]


@pytest.mark.parametrize("form", PLAIN)
@pytest.mark.parametrize("periodic", [False, True])
def test_plain_bricks_match_cpu_fp32(gpu, form, periodic):
    import torch
    import torch.nn.functional as F
    from taichi_lbm3d_amd import surrogate as sg
    from test_gpu_surrogate import torch_weight
    n, d, h, w, cin, cout, ct = form
    assert tiles_of(n, d, h, w, cout)[0] == ct
    if (cin // 16) % 2:
        assert tiles_of(n, d, h, w, cout)[1] > 768 * ct * 16 // cout  # more bricks than workgroups
    x, wt, b = make_case((n, d, h, w, cin, cout, 3), 50)
    y = sg.conv_fwd(x.to(gpu), wt.to(gpu), b.to(gpu), cout, 3, False, periodic=periodic)
    packed, _ = sg.pack_weights(wt.float().to(gpu), False)
    assert torch.equal(y, sg.conv_fwd_packed(x.to(gpu), packed, b.to(gpu), cout, False, periodic=periodic))
    if periodic:
        xt = x.float().permute(0, 4, 1, 2, 3)
        for dim, m in ((2, d), (3, h), (4, w)):
            xt = xt.index_select(dim, torch.tensor([m - 1] + list(range(m)) + [0]))
        ref = F.conv3d(xt, torch_weight(wt, cin, cout, 3), b).permute(0, 2, 3, 4, 1)
    else:
        ref = cpu_conv(x, wt, b, cin, cout, 3, False)
    # FP32 accumulation of exact bf16 products on both sides, then one rounding to bf16 (half of 2^-8 of the value)
    err = (y.float().cpu() - ref).abs()
    assert (err <= 2 ** -8 * ref.abs() + 1e-4 * ref.abs().max()).all()


@pytest.mark.parametrize("form", [(2, 34, 46, 50, 64, 64, 4), (1, 34, 42, 50, 64, 128, 4), (2, 34, 46, 50, 64, 32, 2),
                                  (2, 34, 60, 50, 80, 16, 1), (2, 34, 60, 50, 112, 32, 2), (1, 34, 42, 50, 16, 64, 4)])
@pytest.mark.parametrize("periodic", [False, True])
def test_pooled_bricks(gpu, form, periodic):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout, ct = form
    assert cin == 16 or tiles_of(n, d, h, w, cout)[0] == ct
    (x,), wt, b, _ = tensors(gpu, [(n, d, h, w)], [cin], cout, 51)
    with torch.no_grad():
        y, p = sg.conv3d_pool(x, wt, b, periodic)
        ref = sg.conv3d(x, wt, b, 3, True, periodic=periodic)
    assert torch.equal(y, ref) and torch.equal(p, pool(ref))


# n, d, h, w, c_low, c_skip, cout, channel tiles (0: marching)
UPSAMPLED = [(2, 34, 46, 50, 64, 32, 32, 2), (2, 34, 46, 50, 128, 64, 64, 4), (1, 34, 42, 50, 64, 32, 128, 4),
             (2, 34, 60, 50, 64, 16, 32, 2), (1, 6, 10, 18, 16, 32, 48, 0), (1, 12, 20, 34, 32, 32, 48, 1),
             (2, 4, 8, 16, 48, 16, 96, 1), (1, 34, 42, 50, 48, 16, 96, 2), (1, 6, 10, 18, 16, 16, 96, 0)]


@pytest.mark.parametrize("form", UPSAMPLED)
@pytest.mark.parametrize("periodic", [False, True])
def test_upsampled_bricks(gpu, form, periodic):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cl, cs, cout, ct = form
    assert ct == 0 or tiles_of(n, d, h, w, cout)[0] == ct
    (low, skip), wt, b, _ = tensors(gpu, [(n, d // 2, h // 2, w // 2), (n, d, h, w)], [cl, cs], cout, 52)
    with torch.no_grad():
        y = sg.conv3d_up(low, skip, wt, b, periodic)
        ref = sg.conv3d(torch.cat([up(low), skip], -1), wt, b, 3, True, periodic=periodic)
    assert torch.equal(y, ref)


# n, d, h, w, c_low, c_skip, channels of the gradient, channel tiles (0: marching, 4 tiles and fewer)
SPLIT = [(1, 34, 42, 50, 64, 32, 64, 2), (1, 34, 42, 50, 128, 64, 64, 4), (1, 6, 10, 18, 128, 64, 64, 1),
         (2, 34, 60, 50, 32, 16, 80, 1), (2, 34, 60, 50, 64, 32, 112, 2), (1, 6, 18, 34, 32, 32, 16, 0),
         (1, 40, 16, 16, 32, 32, 16, 0), (1, 6, 18, 34, 32, 16, 16, 0), (2, 6, 18, 34, 64, 32, 32, 0)]


@pytest.mark.parametrize("form", SPLIT)
def test_split_data_gradients_and_the_order_of_their_sums(gpu, form):
    """The low part is the sum of each block of 8 of the plain data gradient's BF16 values, in
    FP32: first the two planes, then the four (y, x) in turn; rounded once."""
    import torch
    from taichi_lbm3d_amd import _lib
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cl, cs, cout, ct = form
    assert ct == 0 or tiles_of(n, d, h, w, cl + cs)[0] == ct
    (g,), wt, _, _ = tensors(gpu, [(n, d, h, w)], [cout], cl + cs, 53)
    wt = torch.randn((cout, _lib.lib().cdll.lbm3d_conv_kpad(cl + cs, 3)), device=gpu) * 0.1
    _, flipped = sg.pack_weights(wt, True)
    full = sg.conv_fwd_packed(g, flipped, None, cl + cs, False)
    d_low = torch.empty((n, d // 2, h // 2, w // 2, cl), dtype=torch.bfloat16, device=gpu)
    d_skip = torch.empty((n, d, h, w, cs), dtype=torch.bfloat16, device=gpu)
    _lib.lib().call("lbm3d_conv3d_dgrad_up", torch.cuda.current_stream().cuda_stream, g.data_ptr(), flipped.data_ptr(),
                    d_low.data_ptr(), d_skip.data_ptr(), n, d, h, w, cl, cs, cout)
    assert torch.equal(d_skip, full[..., cl:])
    part = full[..., :cl].float()
    z = part[:, ::2] + part[:, 1::2]
    s = ((z[:, :, ::2, ::2] + z[:, :, ::2, 1::2]) + z[:, :, 1::2, ::2]) + z[:, :, 1::2, 1::2]
    assert torch.equal(d_low, s.to(torch.bfloat16))
