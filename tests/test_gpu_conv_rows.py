"""3x3x3 convolutions with weights as rows where a workgroup stages them (one channel tile, more
than 48 input channels or a multiple of 64 outputs): the packed weights' results bit for bit,
over one and several bricks a workgroup, even and odd numbers of 16-channel chunks, and times
of the same order."""
import pytest

from test_gpu_unet_blocks import tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [(1, 1, 1, 1, 64, 16), (1, 5, 9, 17, 80, 48), (2, 24, 24, 24, 64, 64),
                                  (1, 40, 33, 50, 96, 32), (2, 34, 60, 50, 112, 16), (2, 34, 60, 50, 128, 16),
                                  (1, 6, 10, 18, 32, 64)])
@pytest.mark.parametrize("periodic", [False, True])
def test_rows_give_the_packed_weights_results(gpu, form, periodic):
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    n, d, h, w, cin, cout = form
    (x,), wt, b, _ = tensors(gpu, [(n, d, h, w)], [cin], cout, 14)
    rows = sg.conv_fwd(x, wt.to(torch.bfloat16), b, cout, 3, True, periodic)
    assert torch.equal(rows, sg.conv_fwd_packed(x, sg.pack_weights(wt, False)[0], b, cout, True, periodic))


def test_rows_cost_little_more_than_packed_weights(gpu):
    """80 -> 80 channels at 2 x 64^3 (about 280 us packed; 296 with rows, 467 with every wave fetching them)."""
    import torch
    from taichi_lbm3d_amd import surrogate as sg
    (x,), wt, b, _ = tensors(gpu, [(2, 64, 64, 64)], [80], 80, 15)
    wb, wp = wt.to(torch.bfloat16), sg.pack_weights(wt, False)[0]

    def best(f):
        times = []
        for _ in range(10):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            f()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    packed = best(lambda: sg.conv_fwd_packed(x, wp, b, 80, True))
    assert best(lambda: sg.conv_fwd(x, wb, b, 80, 3, True)) < 1.35 * packed
