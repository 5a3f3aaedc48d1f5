"""Folds of partial sums at the edges of their groups: bias gradients over 1 to
2048 sets and weight gradients of every block size, with whole numbers, whose
FP32 sums are exact in any order."""
import pytest

pytestmark = pytest.mark.gpu

# voxels, channels: a set holds 16,384 / channels voxels up to 2048 sets, larger ones beyond
SUMS = [(1, 8), (7, 16), (2048, 16), (16 * 1024, 16), (16 * 1024 + 1, 16), (17 * 512, 32), (255 * 64, 256),
        (256 * 1024, 16), (256 * 1024 + 3, 16), (300 * 2048, 8), (2048 * 1024 + 5000, 16)]


@pytest.mark.parametrize("vox,c", SUMS)
def test_bias_gradient_sums_are_exact_for_whole_numbers(gpu, vox, c):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    gen = torch.Generator(device=gpu).manual_seed(vox)
    g = torch.randint(-3, 4, (vox, c), generator=gen, device=gpu).to(torch.bfloat16)
    dz, db = sg.relu_bias_grad(g, None)
    assert torch.equal(dz, g)
    assert torch.equal(db.double(), g.double().sum(0))  # at most 3 * 2.2e6 < 2^24


# n, d, h, w, cin, cout, ks: one set, more than 16 and 256 sets of 256, 7,168, 13,824
# and more elements, and (1x1x1) more than 4096
@pytest.mark.parametrize("form", [(1, 2, 8, 16, 16, 16, 3), (1, 9, 33, 40, 16, 16, 3), (1, 40, 48, 64, 16, 16, 3),
                                  (1, 24, 40, 48, 16, 32, 3), (1, 10, 24, 40, 32, 32, 3), (1, 1, 3, 5, 16, 16, 1),
                                  (1, 72, 80, 96, 16, 16, 1)])
def test_weight_gradient_folds_are_exact_for_whole_numbers(gpu, form):
    import torch
    import torch.nn.functional as F
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout, ks = form
    gen = torch.Generator(device=gpu).manual_seed(d)
    x = torch.randint(-1, 2, (n, d, h, w, cin), generator=gen, device=gpu).to(torch.bfloat16)
    g = torch.randint(-1, 2, (n, d, h, w, cout), generator=gen, device=gpu).to(torch.bfloat16)
    dw = sg.conv_wgrad(x, g, ks)
    p = ks // 2
    xp = F.pad(x.double(), (0, 0, p, p, p, p, p, p))
    gt = g.double().reshape(-1, cout).t().contiguous()
    for tap in range(ks ** 3):
        z, y, c = tap // ks ** 2, tap // ks % ks, tap % ks
        want = gt @ xp[:, z:z + d, y:y + h, c:c + w].reshape(-1, cin)
        assert torch.equal(dw[:, tap * cin:(tap + 1) * cin].double(), want), tap
    assert not dw[:, ks ** 3 * cin:].any()
