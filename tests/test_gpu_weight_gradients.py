"""Weight gradients at the edges of their bricks and folds, against FP64 sums of
the same bf16 products, and the order of the sums: a set's bricks and the number
of sets alone fix it, so that the upsampled form equals the plain one."""
import pytest

pytestmark = pytest.mark.gpu

# n, d, h, w, cin, cout, ks: one brick and its remainders, one and two output
# channel tiles a workgroup, up to 16, 256, 4,096 and more sets to fold, with a
# few and with many elements
FORMS = [
    (1, 1, 1, 1, 16, 16, 3), (1, 3, 9, 17, 16, 16, 3), (1, 2, 8, 16, 16, 32, 3), (2, 3, 10, 18, 48, 48, 3),
    (1, 5, 17, 33, 32, 64, 3), (1, 6, 24, 48, 128, 128, 3), (1, 40, 48, 64, 16, 16, 3), (2, 9, 24, 40, 64, 32, 3),
    (1, 1, 1, 1, 16, 16, 1), (1, 3, 9, 17, 32, 16, 1), (1, 36, 64, 80, 16, 16, 1), (1, 130, 130, 130, 16, 16, 1),
]


@pytest.mark.parametrize("form", FORMS)
def test_weight_gradient_matches_fp64(gpu, form):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout, ks = form
    gen = torch.Generator(device=gpu).manual_seed(7)
    x = torch.randn((n, d, h, w, cin), generator=gen, device=gpu).to(torch.bfloat16)
    g = torch.randn((n, d, h, w, cout), generator=gen, device=gpu).to(torch.bfloat16)
    dw = sg.conv_wgrad(x, g, ks)
    xp = x.double()
    if ks == 3:
        xp = torch.zeros((n, d + 2, h + 2, w + 2, cin), dtype=torch.float64, device=gpu)
        xp[:, 1:-1, 1:-1, 1:-1] = x.double()
    gd = g.double().reshape(-1, cout)
    ref, size = torch.zeros_like(dw, dtype=torch.float64), torch.zeros_like(dw, dtype=torch.float64)
    for t in range(ks ** 3):
        a, b, c = (t // 9, t // 3 % 3, t % 3) if ks == 3 else (0, 0, 0)
        s = xp[:, a:a + d, b:b + h, c:c + w].reshape(-1, cin)
        ref[:, t * cin:(t + 1) * cin] = gd.t() @ s
        size[:, t * cin:(t + 1) * cin] = gd.abs().t() @ s.abs()
    # FP32 sums of exact products: a chain of at most 64 MFMAs of 32 terms and three levels of 16
    # terms, each rounding within 2^-24 of the running sum of magnitudes
    assert ((dw.double() - ref).abs() <= (64 + 48) * 2.0 ** -24 * size).all()
    assert (dw[:, ks ** 3 * cin:] == 0).all()
    assert torch.equal(dw, sg.conv_wgrad(x, g, ks))


@pytest.mark.parametrize("channels", [8, 16, 128])
@pytest.mark.parametrize("voxels", [1, 100, 70000])
def test_bias_gradient_matches_fp64(gpu, channels, voxels):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    gen = torch.Generator(device=gpu).manual_seed(8)
    g = torch.randn((voxels, channels), generator=gen, device=gpu).to(torch.bfloat16)
    y = torch.randn((voxels, channels), generator=gen, device=gpu).relu().to(torch.bfloat16)
    dz, db = sg.relu_bias_grad(g, y)
    assert torch.equal(dz, g * (y > 0))
    want = dz.double().sum(0)
    # a thread adds at most 16 terms, a block 512, then three levels of 16
    assert ((db.double() - want).abs() <= (16 + 512 + 48) * 2.0 ** -24 * dz.double().abs().sum(0) + 1e-30).all()
