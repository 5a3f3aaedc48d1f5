"""Warm-start surrogate: a 3-D U-Net that predicts steady (v, rho - 1) from the
geometry, on the hand-written BF16 MFMA convolutions of conv3d.hip.

No reference counterpart: the reference always starts at rest (init,
SP:160-170).  The network's prediction initialises f at equilibrium through
init_from_macros (a warm start); a cold start stays the fallback.

Network: 4 levels of 16-32-64-128 channels, two 3x3x3 convolutions with ReLU
per level, 2x2x2 max pooling down, nearest-neighbour upsampling and channel
concatenation up, a 1x1x1 head.  Activations and weights are BF16 in the
kernels, accumulation FP32; master weights and Adam state are FP32.  Tensors
are channels-last (N, X, Y, Z, C) throughout.

Inputs (2 channels): solid mask, Euclidean distance to the nearest solid cell
/ DIST_SCALE.  Outputs (4 channels): (vx, vy, vz) / (fx / nu_eff) and
(rho - 1) / (fx * RHO_SCALE): fields in units of the body force, so one
network serves any small force.
"""
from __future__ import annotations

import math

import numpy as np

from . import _lib

CIN_PAD = 16        # input channels are zero-padded to the kernels' multiple of 16
HEAD_PAD = 16       # the 4 output channels are computed as 16 (12 zero rows)
DIST_SCALE = 8.0
RHO_SCALE = 100.0
CHANNELS = (16, 32, 64, 128)
BORDER = 16         # cells next to a volume face that the loss ignores and inference pads around


def _torch():
    import torch
    return torch


def _vp(t):
    return t.data_ptr()


def _stream(dev):
    return _lib.raw_stream(_torch().cuda.current_device() if dev.index is None else dev.index)


def _operand(t):
    """t contiguous and starting on 16 bytes, as the kernels that load straight to LDS read it."""
    if t.is_contiguous() and not t.data_ptr() & 15:
        return t
    return t.clone(memory_format=_torch().contiguous_format)


# ---- the convolution as an autograd function ----------------------------------------------

CONV_RELU, CONV_PERIODIC = 1, 2  # lbm3d_conv3d_fwd flags


def conv_fwd(x, w_bf16, bias, cout, ks, relu, periodic=False):
    """x (N,X,Y,Z,Cin) bf16 contiguous, w_bf16 (cout, kpad) bf16 -> (N,X,Y,Z,cout) bf16.
    periodic: each volume is one period of a periodic field (taps wrap instead of
    reading zero padding)."""
    torch = _torch()
    n, d, h, wd, cin = x.shape
    x, w_bf16 = _operand(x), _operand(w_bf16)
    y = torch.empty((n, d, h, wd, cout), dtype=torch.bfloat16, device=x.device)
    flags = (CONV_RELU if relu else 0) | (CONV_PERIODIC if periodic else 0)
    _lib.lib().call("lbm3d_conv3d_fwd", _stream(x.device), _vp(x), _vp(w_bf16),
                    _vp(bias) if bias is not None else None, _vp(y), n, d, h, wd, cin, cout, ks, flags)
    return y


def conv_dgrad(dy, w_bf16, cin, ks):
    torch = _torch()
    dy = _operand(dy)
    n, d, h, wd, cout = dy.shape
    lib = _lib.lib()
    kpad_t = lib.cdll.lbm3d_conv_kpad(cout, ks)
    wt = torch.empty((cin, kpad_t), dtype=torch.bfloat16, device=dy.device)
    s = _stream(dy.device)
    lib.call("lbm3d_conv3d_wflip", s, _vp(w_bf16), _vp(wt), cin, cout, ks)
    dx = torch.empty((n, d, h, wd, cin), dtype=torch.bfloat16, device=dy.device)
    lib.call("lbm3d_conv3d_dgrad", s, _vp(dy), _vp(wt), _vp(dx), n, d, h, wd, cin, cout, ks)
    return dx


def pack_weights(w, flip: bool):
    """FP32 or BF16 3x3x3 weights (cout, kpad) as BF16 MFMA fragments: (forward, data
    gradient or None)."""
    torch = _torch()
    if w.dim() != 2 or w.dtype not in (torch.float32, torch.bfloat16) or not w.is_contiguous():
        raise ValueError("weights to pack have to be contiguous FP32 or BF16 (cout, kpad), got "
                         f"{tuple(w.shape)} {w.dtype}")
    cout, kpad = w.shape
    cin = kpad // 27 // 16 * 16
    n = 28 * cin * cout  # lbm3d_conv3d_packed_elements
    buf = torch.empty(n * (2 if flip else 1), dtype=torch.bfloat16, device=w.device)
    at = buf.data_ptr()
    _lib.lib().call("lbm3d_conv3d_wpack_bf16" if w.dtype == torch.bfloat16 else "lbm3d_conv3d_wpack", _stream(w.device),
                    w.data_ptr(), at, at + 2 * n if flip else None, cin, cout)
    return (buf[:n], buf[n:]) if flip else (buf, None)


def pack_layers(layers):
    """pack_weights of several (w, flip), all FP32, in one launch."""
    torch = _torch()
    for w, _ in layers:
        if w.dim() != 2 or w.dtype != torch.float32 or not w.is_contiguous() or w.device != layers[0][0].device:
            raise ValueError("weights to pack have to be contiguous FP32 (cout, kpad) on one device, got "
                             f"{tuple(w.shape)} {w.dtype}")
    return _pack_layers(layers) if layers else []


def _pack_layers(layers):
    torch = _torch()
    items, spans, total, dev = (_lib.ConvPack * len(layers))(), [], 0, layers[0][0].device
    for it, (w, flip) in zip(items, layers):
        cout, kpad = w.shape
        it.cout, it.cin = cout, kpad // 27 // 16 * 16
        n = 28 * it.cin * cout  # lbm3d_conv3d_packed_elements
        spans.append((total, n, flip))
        total += n * (2 if flip else 1)
    buf = torch.empty(total, dtype=torch.bfloat16, device=dev)
    for it, (w, _), (at, n, flip) in zip(items, layers, spans):
        it.w, it.wp = w.data_ptr(), buf.data_ptr() + 2 * at
        it.wt = it.wp + 2 * n if flip else None
    _lib.lib().call("lbm3d_conv3d_wpack_many", _stream(dev), len(layers), items)
    return [(buf[at:at + n], buf[at + n:at + 2 * n] if flip else None) for at, n, flip in spans]


def conv_fwd_packed(x, wp, bias, cout, relu, periodic=False):
    """conv_fwd with ks = 3 and the fragments of pack_weights."""
    if wp.numel() != 28 * x.shape[-1] * cout:
        raise ValueError(f"the packed weights are not those of a layer {x.shape[-1]} -> {cout}")
    return _conv_fwd_packed(_operand(x), wp, bias, cout, relu, periodic)


def _conv_fwd_packed(x, wp, bias, cout, relu, periodic=False):
    torch = _torch()
    n, d, h, wd, cin = x.shape
    y = torch.empty((n, d, h, wd, cout), dtype=torch.bfloat16, device=x.device)
    flags = (CONV_RELU if relu else 0) | (CONV_PERIODIC if periodic else 0)
    _lib.lib().call("lbm3d_conv3d_fwd_packed", _stream(x.device), _vp(x), _vp(wp),
                    _vp(bias) if bias is not None else None, _vp(y), n, d, h, wd, cin, cout, flags)
    return y


def conv_wgrad(x, dy, ks):
    return _conv_wgrad(_operand(x), _operand(dy), ks)


def _conv_wgrad(x, dy, ks):
    torch = _torch()
    n, d, h, wd, cin = x.shape
    cout = dy.shape[-1]
    lib = _lib.lib()
    kpad = lib.cdll.lbm3d_conv_kpad(cin, ks)
    ws_bytes = lib.size("lbm3d_conv3d_wgrad_workspace_bytes", n, d, h, wd, cin, cout, ks)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
    dw = torch.empty((cout, kpad), dtype=torch.float32, device=x.device)
    lib.call("lbm3d_conv3d_wgrad", _stream(x.device), _vp(x), _vp(dy), _vp(dw), n, d, h, wd, cin, cout, ks,
             _vp(ws), ws_bytes)
    return dw


def relu_bias_grad(g, y=None):
    """(dz, db) for y = relu(z) with z = conv + b: dz = g * (y > 0) (or g
    without y) in BF16 and db = sum of dz over the voxels in FP32, in one pass
    (lbm3d_relu_bias_grad).  g, y: (..., C) BF16 channels-last."""
    torch = _torch()
    g = g.contiguous()
    c = g.shape[-1]
    vox = g.numel() // c
    lib = _lib.lib()
    ws_bytes = lib.size("lbm3d_relu_bias_grad_workspace_bytes", vox, c)
    ws = torch.empty(max(ws_bytes, 4), dtype=torch.uint8, device=g.device)
    dz = torch.empty_like(g)
    db = torch.empty(c, dtype=torch.float32, device=g.device)
    lib.call("lbm3d_relu_bias_grad", _stream(g.device), _vp(g), _vp(y.contiguous()) if y is not None else None,
             _vp(dz), _vp(db), vox, c, _vp(ws), ws_bytes)
    return dz, db


def relu_pool_grad(g, g_pool, y, pooled):
    """(dz, db) of relu_bias_grad for a layer whose output y was also pooled:
    g_pool is the gradient of its 2x2x2 maximum `pooled`, shared evenly among
    the voxels that attain it and added to g in BF16 (lbm3d_relu_pool_grad)."""
    torch = _torch()
    n, d, h, wd, c = y.shape
    lib = _lib.lib()
    ws_bytes = lib.size("lbm3d_relu_bias_grad_workspace_bytes", n * d * h * wd, c)
    ws = torch.empty(max(ws_bytes, 4), dtype=torch.uint8, device=g.device)
    share = torch.empty_like(pooled)
    dz = torch.empty_like(y)
    db = torch.empty(c, dtype=torch.float32, device=g.device)
    lib.call("lbm3d_relu_pool_grad", _stream(g.device), _vp(g), _vp(y), _vp(pooled), _vp(g_pool), _vp(dz), _vp(db),
             n, d, h, wd, c, _vp(share), _vp(ws), ws_bytes)
    return dz, db


def head_fwd(x, w_bf16, bias):
    """The head's 4 channels, rounded to BF16, in FP32 (lbm3d_conv_head_fwd)."""
    torch = _torch()
    cin = x.shape[-1]
    y = torch.empty(x.shape[:-1] + (4,), dtype=torch.float32, device=x.device)
    _lib.lib().call("lbm3d_conv_head_fwd", _stream(x.device), _vp(x), _vp(w_bf16), _vp(bias), _vp(y), x.numel() // cin,
                    cin)
    return y


def head_fields(x, w_bf16, bias, solid, origin, scale_v, scale_rho, rho_one):
    """(rho, v) of the box at `origin`, of `solid`'s shape, from one volume x
    (X, Y, Z, C) of the last layer's output (lbm3d_conv_head_fields).  solid is any
    mask, nonzero = solid."""
    torch = _torch()
    x, solid = x.contiguous(), _solid_bytes(solid, x.device, "head_fields")
    rho = torch.empty(solid.shape, dtype=torch.float32, device=x.device)
    v = torch.empty(tuple(solid.shape) + (3,), dtype=torch.float32, device=x.device)
    box = [(_lib.ctypes.c_int32 * 3)(*t) for t in (x.shape[:3], origin, solid.shape)]
    _lib.lib().call("lbm3d_conv_head_fields", _stream(x.device), _vp(x), _vp(w_bf16), _vp(bias), _vp(solid), _vp(rho),
                    _vp(v), *box, x.shape[-1], scale_v, scale_rho, int(rho_one))
    return rho, v


def head_grad(g):
    """(dz, db) of the head's 16 channels from the gradient of its 4 outputs (lbm3d_conv_head_grad)."""
    torch = _torch()
    vox = g.numel() // 4
    lib = _lib.lib()
    ws_bytes = lib.size("lbm3d_relu_bias_grad_workspace_bytes", vox, HEAD_PAD)
    ws = torch.empty(max(ws_bytes, 4), dtype=torch.uint8, device=g.device)
    dz = torch.empty(g.shape[:-1] + (HEAD_PAD,), dtype=torch.bfloat16, device=g.device)
    db = torch.empty(HEAD_PAD, dtype=torch.float32, device=g.device)
    lib.call("lbm3d_conv_head_grad", _stream(g.device), _vp(g), _vp(dz), _vp(db), vox, _vp(ws), ws_bytes)
    return dz, db


def _bf16(t):
    return t.contiguous().to(_torch().bfloat16)


def _check_layer(x, cin, w, b, ks, given=None):
    """The kernels take a layer's shapes from x: its weights have to be of them, or they are read past their end."""
    k, shape = ks ** 3 * cin, w.shape
    kpad = (k + 31) // 32 * 32  # lbm3d_conv_kpad
    if len(shape) != 2 or shape[1] != kpad:
        raise ValueError(f"a layer of {cin} input channels takes weights (cout, {kpad}), got {tuple(shape)}")
    device = x.get_device()
    if b is not None and (b.numel() < shape[0] or b.get_device() != device):
        raise ValueError(f"{shape[0]} output channels take as many biases on {x.device}, got {b.numel()} on {b.device}")
    if w.get_device() != device:
        raise ValueError(f"the weights have to be on the input's device {x.device}")
    if given is not None and given[0].numel() != 28 * cin * shape[0]:
        raise ValueError(f"the packed weights are not those of a layer {cin} -> {shape[0]}")


def _check_volume(x, what):
    if x.dim() != 5 or x.dtype != _torch().bfloat16:
        raise ValueError(f"{what} has to be (N, X, Y, Z, C) bfloat16, got {tuple(x.shape)} {x.dtype}")


def _make_conv_functions():
    torch = _torch()

    def packed(w, flip, given):  # given: the layer's fragments from pack_layers, or None
        if given is not None and (not flip or given[1] is not None):
            return given[0], given[1] if flip else None
        return pack_weights((w if w.dtype == torch.float32 else w.to(torch.bfloat16)).contiguous(), flip)

    class Conv3dMFMA(torch.autograd.Function):
        """y = act(conv3d(x, w) + b) with the MFMA kernels in both directions."""

        @staticmethod
        def forward(ctx, x, w, b, ks, relu, need_dx, periodic, given):
            x = _operand(x)
            # Weights that are not FP32 are read as rows where the kernels keep them in registers (few channels):
            # BF16 ones 16 -> 16 channels at 6^3 voxels 13.5 us without the pass that packs them, 20 with it; but
            # 128 -> 128 at 24^3 48 us against 30.
            flip = need_dx and ctx.needs_input_grad[0]
            ctx.packed = ks == 3 and (given is not None or w.dtype == torch.float32
                                      or max(x.shape[-1], w.shape[0] if flip else 0) > 48)
            if ctx.packed:
                wp, wb = packed(w, flip, given)
                y = _conv_fwd_packed(x, wp, b, w.shape[0], relu, periodic)
            else:
                wb = w.to(torch.bfloat16).contiguous()
                y = conv_fwd(x, wb, b, w.shape[0], ks, relu, periodic)
            ctx.save_for_backward(x, wb, y if relu else None)
            ctx.ks, ctx.relu, ctx.need_dx, ctx.periodic = ks, relu, need_dx, periodic
            return y

        @staticmethod
        def backward(ctx, gy):
            if ctx.periodic:
                raise NotImplementedError("periodic convolutions are forward-only (inference)")
            x, wb, y = ctx.saved_tensors
            g, db = relu_bias_grad(_bf16(gy), y if ctx.relu else None)
            dw = _conv_wgrad(x, g, ctx.ks)
            dx = None
            if ctx.need_dx and ctx.needs_input_grad[0]:
                dx = (_conv_fwd_packed(g, wb, None, x.shape[-1], False) if ctx.packed
                      else conv_dgrad(g, wb, x.shape[-1], ctx.ks))
            return dx, dw, db, None, None, None, None, None

    class ConvPool(torch.autograd.Function):
        """(y, 2x2x2 max of y) for y = relu(conv3d(x, w) + b), 3x3x3."""

        @staticmethod
        def forward(ctx, x, w, b, periodic, given):
            x = _operand(x)
            n, d, h, wd, cin = x.shape
            cout = w.shape[0]
            wp, wt = packed(w, ctx.needs_input_grad[0], given)
            y = torch.empty((n, d, h, wd, cout), dtype=torch.bfloat16, device=x.device)
            pooled = torch.empty((n, d // 2, h // 2, wd // 2, cout), dtype=torch.bfloat16, device=x.device)
            _lib.lib().call("lbm3d_conv3d_fwd_pool", _stream(x.device), _vp(x), _vp(wp), _vp(b), _vp(y), _vp(pooled),
                            n, d, h, wd, cin, cout, CONV_RELU | (CONV_PERIODIC if periodic else 0))
            ctx.save_for_backward(x, wt, y, pooled)
            ctx.periodic = periodic
            return y, pooled

        @staticmethod
        def backward(ctx, gy, g_pool):
            if ctx.periodic:
                raise NotImplementedError("periodic convolutions are forward-only (inference)")
            x, wt, y, pooled = ctx.saved_tensors
            g, db = relu_pool_grad(_bf16(gy), _bf16(g_pool), y, pooled)
            dw = _conv_wgrad(x, g, 3)
            dx = _conv_fwd_packed(g, wt, None, x.shape[-1], False) if ctx.needs_input_grad[0] else None
            return dx, dw, db, None, None

    class ConvUp(torch.autograd.Function):
        """relu(conv3d(cat(upsampled low, skip), w) + b), 3x3x3, without the concatenation."""

        @staticmethod
        def forward(ctx, low, skip, w, b, periodic, given):
            low, skip = _operand(low), _operand(skip)
            n, d, h, wd, c_skip = skip.shape
            cout = w.shape[0]
            wp, wt = packed(w, ctx.needs_input_grad[0] or ctx.needs_input_grad[1], given)
            y = torch.empty((n, d, h, wd, cout), dtype=torch.bfloat16, device=skip.device)
            _lib.lib().call("lbm3d_conv3d_fwd_up", _stream(skip.device), _vp(low), _vp(skip), _vp(wp), _vp(b), _vp(y),
                            n, d, h, wd, low.shape[-1], c_skip, cout, CONV_RELU | (CONV_PERIODIC if periodic else 0))
            ctx.save_for_backward(low, skip, wt, y)
            ctx.periodic = periodic
            return y

        @staticmethod
        def backward(ctx, gy):
            if ctx.periodic:
                raise NotImplementedError("periodic convolutions are forward-only (inference)")
            low, skip, wt, y = ctx.saved_tensors
            g, db = relu_bias_grad(_bf16(gy), y)
            n, d, h, wd, c_skip = skip.shape
            c_low, cout = low.shape[-1], g.shape[-1]
            lib, s = _lib.lib(), _stream(g.device)
            kpad = lib.cdll.lbm3d_conv_kpad(c_low + c_skip, 3)
            ws_bytes = lib.size("lbm3d_conv3d_wgrad_workspace_bytes", n, d, h, wd, c_low + c_skip, cout, 3)
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=g.device)
            dw = torch.empty((cout, kpad), dtype=torch.float32, device=g.device)
            lib.call("lbm3d_conv3d_wgrad_up", s, _vp(low), _vp(skip), _vp(g), _vp(dw), n, d, h, wd, c_low, c_skip,
                     cout, _vp(ws), ws_bytes)
            d_low = d_skip = None
            if wt is not None:
                d_low, d_skip = torch.empty_like(low), torch.empty_like(skip)
                lib.call("lbm3d_conv3d_dgrad_up", s, _vp(g), _vp(wt), _vp(d_low), _vp(d_skip), n, d, h, wd, c_low,
                         c_skip, cout)
            return d_low, d_skip, dw, db, None, None

    class Head(torch.autograd.Function):
        """The first 4 channels of a 1x1x1 layer without ReLU, rounded to BF16, as FP32."""

        @staticmethod
        def forward(ctx, x, w, b):
            x = _operand(x)
            wb = w.to(torch.bfloat16).contiguous()
            ctx.save_for_backward(x, wb)
            return head_fwd(x, wb, b)

        @staticmethod
        def backward(ctx, gy):
            x, wb = ctx.saved_tensors
            g, db = head_grad(gy.contiguous())
            dw = _conv_wgrad(x, g, 1)
            dx = conv_dgrad(g, wb, x.shape[-1], 1) if ctx.needs_input_grad[0] else None
            return dx, dw, db

    return Conv3dMFMA, ConvPool, ConvUp, Head


_CONV = None


def _conv_functions():
    global _CONV
    if _CONV is None:
        _CONV = _make_conv_functions()
    return _CONV


def conv3d(x, w, b, ks: int = 3, relu: bool = True, need_dx: bool = True, periodic: bool = False, packed=None):
    """act(conv(x, w) + b); packed: the weights' pack_layers entry, if there is one."""
    _check_layer(x, x.shape[-1], w, b, ks, packed if ks == 3 else None)
    return _conv_functions()[0].apply(x, w, b, ks, relu, need_dx, periodic, packed)


def conv3d_pool(x, w, b, periodic: bool = False, packed=None):
    """(y, its 2x2x2 maximum) of a 3x3x3 layer with ReLU; even extents."""
    _check_volume(x, "the input")
    _check_layer(x, x.shape[-1], w, b, 3, packed)
    return _conv_functions()[1].apply(x, w, b, periodic, packed)


def conv3d_up(low, skip, w, b, periodic: bool = False, packed=None):
    """A 3x3x3 layer with ReLU on the concatenation of `low`, upsampled by 2 (nearest), and `skip`."""
    _check_volume(low, "the low part")
    _check_volume(skip, "the skip part")
    if low.shape[0] != skip.shape[0] or any(a != e // 2 for a, e in zip(low.shape[1:4], skip.shape[1:4])):
        raise ValueError(f"the low part {tuple(low.shape)} does not fit the skip part {tuple(skip.shape)}: "
                         "as many volumes of half the extents")
    if low.device != skip.device:
        raise ValueError(f"the parts are on {low.device} and {skip.device}")
    _check_layer(skip, low.shape[-1] + skip.shape[-1], w, b, 3, packed)
    return _conv_functions()[2].apply(low, skip, w, b, periodic, packed)


def conv_head(x, w, b):
    """The network's head: (..., C) bf16 -> (..., 4) float32."""
    if x.dtype != _torch().bfloat16 or w.shape[0] != HEAD_PAD:
        raise ValueError(f"the head takes bfloat16 and {HEAD_PAD} rows of weights, got {x.dtype}, {tuple(w.shape)}")
    _check_layer(x, x.shape[-1], w, b, 1)
    return _conv_functions()[3].apply(x, w, b)


# ---- the network ------------------------------------------------------------------------------

class UNet3D:
    """Parameters as FP32 master tensors; forward through the MFMA convolutions."""

    def __init__(self, device, seed: int = 0, channels=CHANNELS):
        torch = _torch()
        self.device = device
        self.channels = tuple(channels)
        c1, c2, c3, c4 = self.channels
        specs = [("e1a", CIN_PAD, c1, 3), ("e1b", c1, c1, 3),
                 ("e2a", c1, c2, 3), ("e2b", c2, c2, 3),
                 ("e3a", c2, c3, 3), ("e3b", c3, c3, 3),
                 ("e4a", c3, c4, 3), ("e4b", c4, c4, 3),
                 ("d3a", c4 + c3, c3, 3), ("d3b", c3, c3, 3),
                 ("d2a", c3 + c2, c2, 3), ("d2b", c2, c2, 3),
                 ("d1a", c2 + c1, c1, 3), ("d1b", c1, c1, 3),
                 ("head", c1, HEAD_PAD, 1)]
        self.specs = {name: (cin, cout, ks) for name, cin, cout, ks in specs}
        gen = torch.Generator().manual_seed(seed)
        self.params = {}
        lib = _lib.lib()
        for name, cin, cout, ks in specs:
            kpad = lib.cdll.lbm3d_conv_kpad(cin, ks)
            k = ks ** 3 * cin
            fan_in = k if name != "e1a" else ks ** 3 * 2
            std = math.sqrt(2.0 / fan_in) if name != "head" else math.sqrt(1.0 / fan_in)
            core = torch.randn(cout, ks ** 3, cin, generator=gen) * std
            if name == "e1a":  # only the 2 real input channels carry weights
                core[:, :, 2:] = 0
            w = torch.zeros(cout, kpad)
            w[:, :k] = core.reshape(cout, k)
            if name == "head":
                w[4:] = 0
            self.params[name + ".w"] = w.to(device).requires_grad_(True)
            self.params[name + ".b"] = torch.zeros(cout, device=device).requires_grad_(True)
        # weights that must stay zero: input channels 2..15 of the first layer
        cin, cout, ks = self.specs["e1a"]
        kpad = lib.cdll.lbm3d_conv_kpad(cin, ks)
        keep = torch.zeros(cout, kpad, device=device)
        keep[:, : ks ** 3 * cin] = (torch.arange(ks ** 3 * cin, device=device) % cin < 2).float()
        self._e1a_keep = keep

    def parameters(self):
        return list(self.params.values())

    def _packed(self):
        """Every 3x3x3 layer's weight fragments by name: the data gradient's too where one will be taken."""
        torch = _torch()
        ws = {n: self.params[n + ".w"] for n, (_, _, ks) in self.specs.items() if ks == 3}
        index = next(iter(ws.values())).get_device()
        for n, w in ws.items():
            cin, cout, _ = self.specs[n]
            if w.dtype != torch.float32 or not w.is_contiguous() or w.get_device() != index \
                    or w.shape != (cout, (27 * cin + 31) // 32 * 32):
                return {}  # a layer at a time, each checked by itself
        grad = torch.is_grad_enabled()
        return dict(zip(ws, _pack_layers([(w.detach(), grad and n != "e1a") for n, w in ws.items()])))

    def forward(self, x, periodic: bool = False):
        """x (N,X,Y,Z,16) bf16 with channels 0-1 the inputs -> (N,X,Y,Z,4) float32.
        X, Y, Z must be multiples of 8.  periodic: every volume is one period of a
        periodic geometry, and the convolutions wrap around its faces instead of
        zero padding (forward only)."""
        return conv_head(self._features(x, periodic), self.params["head.w"], self.params["head.b"])

    def _features(self, x, p):
        """The last layer's output before the head, (N,X,Y,Z,C) bf16; p: periodic."""
        packs = self._packed()
        _check_volume(x, "the network's input")
        _check_layer(x, x.shape[-1], self.params["e1a.w"], self.params["e1a.b"], 3)
        # layers that packed fit each other: without the checks of the public calls, 2 us each (a step on 2 x 72^3
        # is bound by the host)
        plain, pooled, joined = (f.apply for f in _conv_functions()[:3]) if packs else (conv3d, conv3d_pool, conv3d_up)

        def conv(name, x, need_dx=True):
            return plain(x, *layer(name), 3, True, need_dx, p, packs.get(name))

        def layer(name):
            return self.params[name + ".w"], self.params[name + ".b"]

        def level(a, b, x, need_dx=True):  # of the encoder: its output, and pooled
            return pooled(conv(a, x, need_dx), *layer(b), p, packs.get(b))

        def up(a, b, low, skip):  # of the decoder
            return conv(b, joined(low, skip, *layer(a), p, packs.get(a)))

        e1, low = level("e1a", "e1b", x, False)
        e2, low = level("e2a", "e2b", low)
        e3, low = level("e3a", "e3b", low)
        d3 = up("d3a", "d3b", conv("e4b", conv("e4a", low)), e3)
        return up("d1a", "d1b", up("d2a", "d2b", d3, e2), e1)

    __call__ = forward

    def zero_head_padding(self):
        """Keep the unused head rows and input-channel weights exactly zero."""
        torch = _torch()
        with torch.no_grad():
            self.params["head.w"][4:] = 0
            self.params["head.b"][4:] = 0
            self.params["e1a.w"].mul_(self._e1a_keep)

    def state_dict(self):
        return {k: v.detach().cpu() for k, v in self.params.items()}

    def load_state_dict(self, sd):
        torch = _torch()
        with torch.no_grad():
            for k, v in sd.items():
                self.params[k].copy_(v.to(self.device))


# ---- inputs and targets -----------------------------------------------------------------------------

def periodic_distance(solid, margin: int = 24, device=None):
    """Euclidean distance of every cell to the nearest solid cell under periodic
    wrap, exact up to `margin` cells and capped there (lbm3d_distance_periodic:
    the separable squared-distance transform, one min-plus pass per axis).
    `solid` is a (X, Y, Z) or (N, X, Y, Z) array or device tensor (nonzero =
    solid); returns a float32 tensor of that shape on the GPU."""
    torch = _torch()
    s = _solid_bytes(solid, device, "periodic_distance")
    dist = torch.empty(s.shape, dtype=torch.float32, device=s.device)
    work = torch.empty_like(dist)
    _lib.lib().call("lbm3d_distance_periodic", _stream(s.device), _vp(s), _vp(dist), _vp(work), *_volumes(s), margin)
    return dist


def _solid_bytes(solid, device, what):
    """A geometry as contiguous int8 on the GPU (nonzero = solid); one-byte types are taken as they are."""
    torch = _torch()
    if torch.is_tensor(solid):
        s = solid if device is None else solid.to(device)
        if s.dtype in (torch.bool, torch.uint8):
            s = s.view(torch.int8)
        elif s.dtype != torch.int8:
            s = (s != 0).to(torch.int8)
    else:
        s = torch.as_tensor(np.asarray(solid) != 0, device=device).to(torch.int8)
    if s.device.type != "cuda":
        raise RuntimeError(f"{what} runs on the GPU (lbm3d_distance_periodic)")
    return s.contiguous()


def _volumes(s):
    return tuple(s.shape) if s.dim() == 4 else (1,) + tuple(s.shape)


def _inputs(s, network: bool, margin: int = 24):
    torch = _torch()
    out = torch.empty(tuple(s.shape) + ((CIN_PAD,) if network else (2,)),
                      dtype=torch.bfloat16 if network else torch.float32, device=s.device)
    work = torch.empty(2 * s.numel(), dtype=torch.float32, device=s.device)
    _lib.lib().call("lbm3d_surrogate_inputs", _stream(s.device), _vp(s), _vp(out), int(network), DIST_SCALE,
                    _vp(work), *_volumes(s), margin)
    return out


def make_inputs(solid, device=None):
    """(X, Y, Z, 2) float32 tensor on the device: solid mask and distance / DIST_SCALE.
    `solid` is a numpy array or a device tensor (nonzero = solid)."""
    return _inputs(_solid_bytes(solid, device, "make_inputs"), False)


def network_inputs(solids):
    """to_network_input(make_inputs(.)) of (N, X, Y, Z) geometries in one go."""
    return _inputs(_solid_bytes(solids, None, "network_inputs"), True)


def make_targets(rho, v, solid, fx, nu_eff):
    """(X, Y, Z, 4) float32 normalised targets; zero on solid cells."""
    fluid = (np.asarray(solid) == 0)[..., None]
    vt = np.asarray(v, np.float32) * (nu_eff / fx)
    rt = (np.asarray(rho, np.float32) - 1.0)[..., None] / (fx * RHO_SCALE)
    return np.where(fluid, np.concatenate([vt, rt], axis=-1), 0.0).astype(np.float32)


def fields_from_prediction(pred, fluid, fx, nu_eff, density=False):
    """Inverse of make_targets on the device: (rho, v, predicted rho) from a
    (X,Y,Z,4) prediction, zero velocity off the fluid.

    By default the warm start takes the predicted velocity with rho = 1, the
    cold start's density.  Every isolated pore keeps its initial mass for good,
    and the steady velocity of a pore scales as 1/rho, so a raw predicted
    density would pin the mean density -- and the permeability, to about the
    prediction's density error -- away from the cold start's.  With
    density=True the returned rho is the predicted density shifted to mean 1
    over the fluid cells: the sample's total mass is the cold start's, and only
    the split of that mass between disconnected pores can differ."""
    torch = _torch()
    p = pred.float()
    fl = fluid.to(p.dtype)
    v = p[..., :3] * (fx / nu_eff) * fl[..., None]
    rho_pred = 1.0 + p[..., 3] * (fx * RHO_SCALE) * fl
    if not density:
        return torch.ones_like(rho_pred), v, rho_pred
    return _mean_one(rho_pred, fluid), v, rho_pred


def _mean_one(rho_pred, fluid):
    """The density shifted to mean 1 over the fluid, 1 elsewhere."""
    fl = fluid.to(rho_pred.dtype)
    n = fl.sum().clamp_min(1.0)
    dev = (rho_pred - 1.0) * fl
    return 1.0 + (dev - dev.sum() / n) * fl


def to_network_input(inp):
    """(N,X,Y,Z,2) float32 tensor -> (N,X,Y,Z,16) bf16 (channels 2..15 zero)."""
    torch = _torch()
    t = torch.zeros(inp.shape[:4] + (CIN_PAD,), dtype=torch.bfloat16, device=inp.device)
    t[..., :2] = inp.to(torch.bfloat16)
    return t


def periodic_pad(t, pad):
    """(X,Y,Z,...) tensor -> (X+lo+hi, ...) per axis, wrapped periodically; `pad`
    is one width for both sides of every axis or a (lo, hi) pair per axis."""
    torch = _torch()
    for axis in range(3):
        lo, hi = pad[axis] if isinstance(pad, (tuple, list)) else (pad, pad)
        n = t.shape[axis]
        idx = (torch.arange(-lo, n + hi, device=t.device) % n)
        t = t.index_select(axis, idx)
    return t


def inference_pads(shape, wrap: bool):
    """(lo, hi) periodic padding per axis for inference: none when the network
    wraps, else BORDER cells before the volume and at least BORDER after it,
    the padded extent a multiple of 8 (the network pools three times)."""
    if wrap:
        return [(0, 0)] * 3
    return [(BORDER, BORDER + (-(n + 2 * BORDER)) % 8) for n in shape]


def _device_solid(solid, device):
    """(X, Y, Z) bool tensor on the device (True = solid) from an array or tensor."""
    torch = _torch()
    if torch.is_tensor(solid):
        return solid.to(device) != 0
    return torch.from_numpy(np.ascontiguousarray(np.asarray(solid) != 0)).to(device)


def predict(net, solids, fx, nu_eff, batch: int = 2, wrap=None, density=False):
    """Warm-start (rho, v) device tensors predicted for periodic geometries of
    one shape (numpy arrays or device tensors), `batch` volumes per forward pass.
    rho is 1, or with density=True the predicted density at mean 1 over the
    fluid (fields_from_prediction).

    wrap=True runs the network's convolutions periodically on the volume itself
    (every extent a multiple of 8): every cell sees its true periodic
    surroundings.  wrap=False pads each volume periodically by at least BORDER
    cells (to a multiple of 8), runs the zero-padded network and keeps the
    centre.  The default wraps when the extents allow it."""
    torch = _torch()
    out = []
    if not len(solids):
        return out
    shape = tuple(solids[0].shape)
    if wrap is None:
        wrap = all(n % 8 == 0 for n in shape)
    if wrap and any(n % 8 for n in shape):
        raise ValueError(f"periodic inference needs extents that are multiples of 8, got {shape}")
    pads = inference_pads(shape, wrap)
    # a network with a forward of its own, or a force per component, goes through its output
    fused = type(net) is UNet3D and isinstance(fx, float) and isinstance(nu_eff, float)
    with torch.no_grad():
        for b0 in range(0, len(solids), batch):
            sol = torch.stack([_device_solid(s, net.device) for s in solids[b0:b0 + batch]])
            if wrap:
                inp = network_inputs(sol)
            else:
                inp = to_network_input(torch.stack([periodic_pad(t, pads) for t in make_inputs(sol)]))
            (X, Y, Z), (px, py, pz) = shape, (p[0] for p in pads)
            if fused:  # the head gives the fields of fields_from_prediction itself
                feat, (w, b) = net._features(inp, wrap), (net.params["head.w"], net.params["head.b"])
                w = w.to(torch.bfloat16).contiguous()
                for i in range(sol.shape[0]):
                    rho, v = head_fields(feat[i], w, b, sol[i], (px, py, pz), fx / nu_eff, fx * RHO_SCALE, not density)
                    out.append((_mean_one(rho, ~sol[i]) if density else rho, v))
                continue
            pred = net(inp, periodic=wrap)
            for i in range(sol.shape[0]):
                core = pred[i, px:px + X, py:py + Y, pz:pz + Z]
                out.append(fields_from_prediction(core, ~sol[i], fx, nu_eff, density)[:2])
    return out
