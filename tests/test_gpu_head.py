"""The 1x1x1 convolution at the edges of its 64-voxel waves, and the network's
head: its output, its gradient and the warm-start fields against the padded
convolution and the tensor operations that they stand for, bit for bit."""
import pytest

from test_gpu_surrogate import cpu_conv, make_case, rand_bf16

pytestmark = pytest.mark.gpu

# n, d, h, w, cin, cout: one voxel, a wave less and more one, a block and one;
# half a K chunk, a whole one, one and a half, many; 1, 2, 3 and 4 output tiles
FORMS = [(1, 1, 1, 1, 16, 16), (1, 7, 9, 1, 16, 16), (1, 1, 5, 13, 48, 32), (1, 1, 1, 257, 32, 48),
         (2, 4, 8, 8, 80, 64), (1, 3, 5, 17, 256, 128), (2, 6, 10, 14, 16, 256)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("relu", [False, True])
def test_pointwise_convolution_matches_cpu_fp32(gpu, form, relu):
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout = form
    x, wt, b = make_case(form + (1,), 50)
    y = sg.conv_fwd(x.to(gpu), wt.to(gpu), b.to(gpu), cout, 1, relu)
    ref = cpu_conv(x, wt, b, cin, cout, 1, relu)
    # FP32 accumulation of exact bf16 products on both sides, then one rounding to bf16 (half of 2^-8 of the value)
    err = (y.float().cpu() - ref).abs()
    assert (err <= 2 ** -8 * ref.abs() + 1e-4 * ref.abs().max()).all()


@pytest.mark.parametrize("form", [(1, 1, 1, 1, 16, 16), (1, 7, 9, 1, 32, 16), (1, 1, 5, 13, 48, 16), (2, 8, 16, 24, 16, 16)])
def test_head_is_the_padded_convolution(gpu, form):
    """Output and gradients of the head equal those of the 16-channel layer and its slice."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    x, wt, b = make_case(form + (1,), 60)
    g = torch.randn(form[:4] + (4,), generator=torch.Generator().manual_seed(61)).to(gpu)
    res = []
    for head in (True, False):
        xi, wi, bi = (t.to(gpu).requires_grad_(True) for t in (x, wt.float(), b))
        y = sg.conv_head(xi, wi, bi) if head else sg.conv3d(xi, wi, bi, 1, False)[..., :4].float()
        y.backward(g)
        res.append((y.detach(), xi.grad, wi.grad, bi.grad))
    for a, c in zip(*res):
        assert a.dtype == c.dtype and torch.equal(a, c)


@pytest.mark.parametrize("extents,origin,core", [((1, 1, 1), (0, 0, 0), (1, 1, 1)), ((5, 7, 13), (0, 0, 0), (5, 7, 13)),
                                                 ((9, 8, 40), (2, 1, 3), (6, 7, 33)), ((24, 16, 16), (16, 0, 8), (8, 16, 8))])
@pytest.mark.parametrize("cin", [16, 48])
@pytest.mark.parametrize("density", [False, True])
def test_head_fields_are_those_of_the_prediction(gpu, extents, origin, core, cin, density):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    x = rand_bf16(extents + (cin,), 70).to(gpu)
    _, wt, b = make_case((1, 1, 1, 1, cin, 16, 1), 71)
    wt, b = wt.to(gpu), b.to(gpu)
    solid = (torch.rand(core, generator=torch.Generator().manual_seed(72)) < 0.4).to(gpu)
    box = tuple(slice(o, o + c) for o, c in zip(origin, core))
    pred = sg.conv_fwd(x[None], wt, b, 16, 1, False)[0][box][..., :4].float()
    fx, nu = 3e-5, 1 / 18
    rho, v, raw = sg.fields_from_prediction(pred, ~solid, fx, nu, density)
    r, u = sg.head_fields(x, wt, b, solid, origin, fx / nu, fx * sg.RHO_SCALE, not density)
    assert torch.equal(u, v) and torch.equal(r, raw if density else rho)


@pytest.mark.parametrize("edge,density", [(16, False), (16, True), (13, False)])
def test_predict_equals_the_network_and_its_fields(gpu, edge, density):
    """predict, wrapped and padded, gives what fields_from_prediction makes of the network's output."""
    import numpy as np
    import torch
    from taichi_lbm3d_amd import surrogate as sg

    class Through(sg.UNet3D):  # a network of its own type goes through its output
        pass

    solids = [np.random.default_rng(80 + i).random((edge,) * 3) < 0.3 for i in range(3)]
    got = sg.predict(sg.UNet3D(gpu, seed=4), solids, 1e-5, 0.1, density=density)
    want = sg.predict(Through(gpu, seed=4), solids, 1e-5, 0.1, density=density)
    for (r, v), (r2, v2) in zip(got, want):
        assert torch.equal(r, r2) and torch.equal(v, v2)


def test_boxes_outside_the_volume_are_refused(gpu):
    import torch
    from taichi_lbm3d_amd import _lib
    from taichi_lbm3d_amd import surrogate as sg
    x, w, b = (torch.zeros(s, dtype=t, device=gpu) for s, t in
               (((4, 4, 4, 16), torch.bfloat16), ((16, 32), torch.bfloat16), ((16,), torch.float32)))
    for origin, core in (((1, 0, 0), (4, 4, 4)), ((0, -1, 0), (2, 2, 2))):
        with pytest.raises(_lib.LbmError):
            sg.head_fields(x, w, b, torch.zeros(core, dtype=torch.bool, device=gpu), origin, 1.0, 1.0, True)
