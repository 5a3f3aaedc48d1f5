"""The surrogate's layers refuse operands that do not fit each other before any kernel reads
them (CPU: no kernel runs here)."""
import pytest
import torch

from taichi_lbm3d_amd import surrogate as sg


def vol(n, x, y, z, c, dtype=torch.bfloat16):
    return torch.zeros((n, x, y, z, c), dtype=dtype)


def weights(cin, cout, ks=3):
    return torch.zeros((cout, (ks ** 3 * cin + 31) // 32 * 32))


@pytest.mark.parametrize("low, skip", [
    (vol(1, 2, 2, 2, 16), vol(1, 4, 4, 6, 16)), (vol(1, 2, 2, 2, 16), vol(1, 8, 4, 4, 16)),
    (vol(1, 2, 2, 2, 16), vol(2, 4, 4, 4, 16)), (vol(2, 2, 2, 2, 16), vol(1, 4, 4, 4, 16)),
    (vol(1, 4, 4, 4, 16), vol(1, 4, 4, 4, 16)),
])
def test_upsampled_parts_have_to_fit(low, skip):
    with pytest.raises(ValueError, match="fit"):
        sg.conv3d_up(low, skip, weights(32, 16), torch.zeros(16))


@pytest.mark.parametrize("w", [weights(16, 16), weights(48, 16), weights(32, 16)[:, :-32], weights(32, 16).view(-1)])
def test_weights_have_to_be_the_input_channels(w):
    b = torch.zeros(16)
    with pytest.raises(ValueError, match="weights"):
        sg.conv3d_up(vol(1, 2, 2, 2, 16), vol(1, 4, 4, 4, 16), w, b)
    with pytest.raises(ValueError, match="weights"):
        sg.conv3d(vol(1, 4, 4, 4, 32), w, b)
    with pytest.raises(ValueError, match="weights"):
        sg.conv3d_pool(vol(1, 4, 4, 4, 32), w, b)
    with pytest.raises(ValueError, match="weights"):
        sg.conv_head(vol(1, 4, 4, 4, 32), torch.zeros(16, 16), b)


def test_biases_and_packed_weights_have_to_be_the_layer():
    x, w, b = vol(1, 4, 4, 4, 16), weights(16, 32), torch.zeros(32)
    with pytest.raises(ValueError, match="biases"):
        sg.conv3d(x, w, b[:16])
    with pytest.raises(ValueError, match="packed"):
        sg.conv3d(x, w, b, packed=(torch.zeros(28 * 16 * 16, dtype=torch.bfloat16), None))
    with pytest.raises(ValueError, match="packed"):
        sg.conv3d_pool(x, w, b, packed=(torch.zeros(28 * 32 * 32, dtype=torch.bfloat16), None))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_volumes_have_to_be_bfloat16(dtype):
    w, b = weights(32, 16), torch.zeros(16)
    for low, skip in ((dtype, torch.bfloat16), (torch.bfloat16, dtype)):
        with pytest.raises(ValueError, match="bfloat16"):
            sg.conv3d_up(vol(1, 2, 2, 2, 16, low), vol(1, 4, 4, 4, 16, skip), w, b)
    with pytest.raises(ValueError, match="bfloat16"):
        sg.conv3d_pool(vol(1, 4, 4, 4, 32, dtype), w, b)
    with pytest.raises(ValueError, match="bfloat16"):
        sg.conv_head(vol(1, 4, 4, 4, 32, dtype), torch.zeros(16, 32), b)


@pytest.mark.parametrize("w", [weights(16, 32).half(), weights(16, 32).double(), weights(16, 32).t(),
                               weights(16, 32)[:, ::2], weights(16, 32).view(-1)])
def test_weights_that_cannot_be_packed_are_refused(w):
    with pytest.raises(ValueError, match="pack"):
        sg.pack_weights(w, True)
    with pytest.raises(ValueError, match="pack"):
        sg.pack_layers([(weights(16, 16), False), (w, True)])


def test_a_convolution_takes_its_own_fragments():
    with pytest.raises(ValueError, match="packed"):
        sg.conv_fwd_packed(vol(1, 4, 4, 4, 32), torch.zeros(28 * 16 * 16, dtype=torch.bfloat16), None, 16, False)


def test_layers_packed_together_are_fp32():
    with pytest.raises(ValueError, match="pack"):
        sg.pack_layers([(weights(16, 32).to(torch.bfloat16), True)])
