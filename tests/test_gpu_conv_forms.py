"""The forward convolution's kernels at the edges of their tiles: the march
along z (up to 48 input channels) and the bricks (more, or 64-channel outputs),
with plain and packed weights, against FP32 CPU convolutions of the same
bf16-rounded operands."""
import numpy as np
import pytest

from test_gpu_surrogate import cpu_conv, make_case, rand_bf16

pytestmark = pytest.mark.gpu

# n, d, h, w, cin, cout: remainders of the 16- and 8-row columns and of the
# bricks, one plane, several runs of planes, 1, 2 and 4 channel tiles per
# workgroup, an odd number of 16-channel chunks
FORMS = [
    (1, 1, 1, 1, 16, 16), (1, 3, 17, 33, 16, 16), (2, 40, 16, 16, 16, 16), (1, 5, 9, 17, 16, 32),
    (1, 3, 9, 15, 16, 64), (1, 4, 8, 16, 32, 16), (2, 9, 10, 18, 32, 32), (1, 7, 10, 18, 48, 16),
    (1, 3, 7, 19, 48, 96), (1, 2, 3, 5, 80, 48), (1, 5, 9, 17, 32, 64), (1, 3, 9, 17, 112, 64),
    (1, 6, 12, 20, 64, 128), (2, 33, 40, 36, 64, 64),
]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("periodic", [False, True])
def test_forward_forms_match_cpu_fp32(gpu, form, periodic):
    import torch
    import torch.nn.functional as F
    from taichi_lbm3d_amd import surrogate as sg
    from test_gpu_surrogate import torch_weight
    n, d, h, w, cin, cout = form
    x, wt, b = make_case(form + (3,), 30)
    y = sg.conv_fwd(x.to(gpu), wt.to(gpu), b.to(gpu), cout, 3, False, periodic=periodic)
    packed, _ = sg.pack_weights(wt.float().to(gpu), False)
    yp = sg.conv_fwd_packed(x.to(gpu), packed, b.to(gpu), cout, False, periodic=periodic)
    assert torch.equal(y, yp)
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


@pytest.mark.parametrize("form", [(1, 3, 9, 17, 16, 48), (1, 4, 6, 5, 64, 32), (1, 2, 3, 5, 80, 16)])
def test_packed_data_gradient_equals_flipped_weights(gpu, form):
    """The packed flipped weights give lbm3d_conv3d_dgrad's result bit for bit."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout = form
    _, wt, _ = make_case(form + (3,), 40)
    gy = rand_bf16((n, d, h, w, cout), 43).to(gpu)
    dx = sg.conv_dgrad(gy, wt.to(gpu), cin, 3)
    _, flipped = sg.pack_weights(wt.float().to(gpu), True)
    assert torch.equal(dx, sg.conv_fwd_packed(gy, flipped, None, cin, False))


def test_packed_weights_round_to_nearest_and_place_every_tap(gpu):
    """Fragment order against its definition, and FP32 weights rounded as torch rounds them."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    cin, cout = 32, 48
    w = torch.zeros(cout, 27 * cin)
    w[:] = torch.randn(w.shape, generator=torch.Generator().manual_seed(3))
    wp, wt = (t.cpu().float().numpy() for t in sg.pack_weights(w.to(gpu), True))
    wb = w.to(torch.bfloat16).float().numpy().reshape(cout, 27, cin)

    def fragments(m, ci_n, co_n):  # m[co][tap][ci]
        out = np.zeros((ci_n // 16, 14, co_n // 16, 64, 8), np.float32)
        for lane in range(64):
            g, r = lane >> 4, lane & 15
            for s in range(14):
                tap = 2 * s + (g >> 1)
                if tap == 27:
                    continue
                for c in range(ci_n // 16):
                    ci = 16 * c + 8 * (g & 1)
                    for t in range(co_n // 16):
                        out[c, s, t, lane] = m[16 * t + r, tap, ci:ci + 8]
        return out.reshape(-1)

    np.testing.assert_array_equal(wp, fragments(wb, cin, cout))
    np.testing.assert_array_equal(wt, fragments(wb.transpose(2, 1, 0)[:, ::-1], cout, cin))


def test_layers_packed_together_equal_layers_packed_alone(gpu):
    """18 layers (more than one launch takes), with and without the flipped weights."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    shapes = [(16, 16), (48, 16), (16, 64), (96, 32), (112, 48), (256, 16)] * 3
    ws = [make_case((1, 1, 1, 1, cin, cout, 3), 60 + i)[1].float().to(gpu) for i, (cin, cout) in enumerate(shapes)]
    many = sg.pack_layers([(w, i % 2 == 0) for i, w in enumerate(ws)])
    for i, (w, (wp, wt)) in enumerate(zip(ws, many)):
        one, flipped = sg.pack_weights(w, True)
        assert torch.equal(wp, one)
        assert torch.equal(wt, flipped) if i % 2 == 0 else wt is None
    assert sg.pack_layers([]) == []
