"""Learned gradient preconditioner: a 4-level U-Net on the HIP kernels of
csrc/unet.hip (BF16 weights and activations, FP32 accumulation on MFMA).

It maps the raw FP32 gradient and the current model of an FWI iteration to an
update direction.  There is no counterpart in the reference: its FWI step
(seistorch/fwi.py with the optimizers of seistorch/optimizer.py) applies the
plain gradient, which remains the fallback whenever the network's direction
does not reduce the misfit.

Architecture (NHWC; C = 32):
    input 2 channels (gradient * gscale, (model - mshift) * mscale), padded to 8
    encoder level l = 0..3 at 1/2^l resolution: conv3x3 -> GELU -> conv3x3 -> GELU
        with C, 2C, 4C, 8C channels, 2x2 average pooling between levels
    bottleneck at 1/16: two conv3x3 + GELU with 8C channels
    decoder l = 3..0: nearest 2x upsampling, concatenation with the encoder
        output of level l, two conv3x3 + GELU back to the level's channels
    head: 1x1 convolution to one FP32 channel
H and W must be multiples of 16.
"""
import math

import numpy as np
import torch

from . import _lib

BASE = 32
IN_CH = 8  # 2 used, padded for 16-byte vector access


def layer_specs(base=BASE):
    """[(name, Cin, Cout)] of the 3x3 convolutions in forward order."""
    ch = [base, 2 * base, 4 * base, 8 * base]
    specs, cin = [], IN_CH
    for l, c in enumerate(ch):
        specs += [(f"enc{l}a", cin, c), (f"enc{l}b", c, c)]
        cin = c
    specs += [("bota", cin, ch[3]), ("botb", ch[3], ch[3])]
    low = ch[3]
    for l in (3, 2, 1, 0):
        specs += [(f"dec{l}a", low + ch[l], ch[l]), (f"dec{l}b", ch[l], ch[l])]
        low = ch[l]
    return specs


class Params:
    """FP32 master parameters in one flat arena (conv weights (Cout, 9*Cin)
    then bias (Cout) per layer, then head weight (C) and bias (1)), plus the
    bf16 copy of the conv weights the kernels read."""

    def __init__(self, device, base=BASE, seed=0):
        self.specs = layer_specs(base)
        self.base = base
        self.off = {}
        o = 0
        for name, cin, cout in self.specs:
            self.off[name] = (o, o + cout * 9 * cin)  # weight, bias offsets
            o += cout * 9 * cin + cout
        self.off["head"] = (o, o + base)
        o += base + 1
        self.n = o
        g = torch.Generator().manual_seed(seed)
        host = torch.zeros(self.n)
        for name, cin, cout in self.specs:
            w0, _ = self.off[name]
            fan_in = 9 * (2 if name == "enc0a" else cin)
            w = torch.randn(cout, 9, cin, generator=g) * math.sqrt(2.0 / fan_in)
            if name == "enc0a":
                w[:, :, 2:] = 0.0  # the padding channels carry nothing
            host[w0:w0 + cout * 9 * cin] = w.reshape(-1)
        h0, _ = self.off["head"]
        host[h0:h0 + base] = torch.randn(base, generator=g) * (0.1 / math.sqrt(base))
        self.master = host.to(device)
        self.bf16 = torch.empty(self.n, dtype=torch.int16, device=device)
        self.refresh_bf16()

    def refresh_bf16(self):
        _lib.call("seis_unet_to_bf16", _lib.ptr(self.master), self.n, _lib.ptr(self.bf16),
                  _lib.stream_of(self.master))

    def weight(self, name, arena=None):
        a = self.master if arena is None else arena
        w0, b0 = self.off[name]
        return a[w0:b0]

    def bias(self, name, arena=None):
        a = self.master if arena is None else arena
        w0, b0 = self.off[name]
        cout = dict((s[0], s[2]) for s in self.specs)[name]
        return a[b0:b0 + cout]

    def wbf16(self, name):
        w0, b0 = self.off[name]
        return self.bf16[w0:b0]

    def head(self, arena=None):
        a = self.master if arena is None else arena
        h0, hb = self.off["head"]
        return a[h0:hb], a[hb:hb + 1]

    def state_dict(self):
        return {"master": self.master.detach().cpu(), "base": self.base}

    def load_state_dict(self, sd):
        self.master.copy_(sd["master"].to(self.master.device))
        self.refresh_bf16()


def _bf(shape, dev):
    return torch.empty(shape, dtype=torch.int16, device=dev)


def _f32(shape, dev):
    return torch.empty(shape, dtype=torch.float32, device=dev)


class UNet:
    """Forward / backward of the network on (N, H, W) gradient and model planes."""

    def __init__(self, params):
        self.p = params

    # -- building blocks -------------------------------------------------
    def _conv(self, x, N, H, W, name, keep):
        _, cin, cout = next(s for s in self.p.specs if s[0] == name)
        dev = x.device
        y = _bf((N, H, W, cout), dev)
        z = _bf((N, H, W, cout), dev) if keep else None
        _lib.call("seis_unet_conv3x3", _lib.ptr(x), N, H, W, cin, _lib.ptr(self.p.wbf16(name)),
                  _lib.ptr(self.p.bias(name)), cout, 1, _lib.ptr(z), _lib.ptr(y), None,
                  _lib.stream_of(x))
        if keep:
            self.saved[name] = (x, z, (N, H, W))
        return y

    def _conv_cat(self, low, skip, N, H, W, name, keep):
        """_conv of the concatenation [2x upsampled low, skip], read in place
        where the kernel can (the channels of low in whole tiles of 64)."""
        c1, c2 = low.shape[-1], skip.shape[-1]
        dev = low.device
        if c1 % 64:
            u = _bf((N, H, W, c1 + c2), dev)
            _lib.call("seis_unet_up_concat", _lib.ptr(low), _lib.ptr(skip), N, H, W, c1, c2,
                      _lib.ptr(u), _lib.stream_of(low))
            return self._conv(u, N, H, W, name, keep)
        _, _, cout = next(s for s in self.p.specs if s[0] == name)
        y = _bf((N, H, W, cout), dev)
        z = _bf((N, H, W, cout), dev) if keep else None
        _lib.call("seis_unet_conv3x3_cat", _lib.ptr(low), c1, _lib.ptr(skip), c2, N, H, W,
                  _lib.ptr(self.p.wbf16(name)), _lib.ptr(self.p.bias(name)), cout, 1,
                  _lib.ptr(z), _lib.ptr(y), _lib.stream_of(low))
        if keep:
            self.saved[name] = ((low, skip), z, (N, H, W))
        return y

    def forward(self, grad, model, scales, keep=False):
        """grad, model (N, H, W) FP32; scales (N, 3) FP32 = (gscale, mscale, mshift).
        Returns the (N, H, W) FP32 direction."""
        N, H, W = grad.shape
        if H % 16 or W % 16:
            raise RuntimeError(f"U-Net input {H}x{W} must be a multiple of 16 in both axes")
        _lib.require_device(grad, model, scales)
        dev = grad.device
        s = _lib.stream_of(grad)
        self.saved = {}
        x = _bf((N, H, W, IN_CH), dev)
        _lib.call("seis_unet_pack_input", _lib.ptr(grad), _lib.ptr(model), N, H, W,
                  _lib.ptr(scales), _lib.ptr(x), s)
        skips, h, w = [], H, W
        for l in range(4):
            x = self._conv(x, N, h, w, f"enc{l}a", keep)
            x = self._conv(x, N, h, w, f"enc{l}b", keep)
            skips.append((x, h, w))
            c = x.shape[-1]
            p = _bf((N, h // 2, w // 2, c), dev)
            _lib.call("seis_unet_avgpool2", _lib.ptr(x), N, h, w, c, _lib.ptr(p), s)
            x, h, w = p, h // 2, w // 2
        x = self._conv(x, N, h, w, "bota", keep)
        x = self._conv(x, N, h, w, "botb", keep)
        for l in (3, 2, 1, 0):
            sk, h, w = skips[l]
            x = self._conv_cat(x, sk, N, h, w, f"dec{l}a", keep)
            x = self._conv(x, N, h, w, f"dec{l}b", keep)
        out = _f32((N, H, W), dev)
        hw, hb = self.p.head()
        _lib.call("seis_unet_head", _lib.ptr(x), N * H * W, self.p.base, _lib.ptr(hw),
                  _lib.ptr(hb), _lib.ptr(out), s)
        if keep:
            self.saved["head_in"] = x
            self.saved["shape"] = (N, H, W)
            self.saved["skip_c"] = [sk.shape[-1] for sk, _, _ in skips]
        return out

    def _wgrad(self, name, dz, gw_arena):
        """Adds the layer's dW and db to the gradient arena (dz: bf16 gradient
        of its pre-activation)."""
        _, cin, cout = next(s for s in self.p.specs if s[0] == name)
        x, _, (N, H, W) = self.saved[name]
        gw, gb = self.p.weight(name, gw_arena), self.p.bias(name, gw_arena)
        low, skip = x if isinstance(x, tuple) else (None, x)
        c1 = low.shape[-1] if low is not None else 0
        n = int(_lib.load().seis_unet_wgrad_workspace(N, H, W, cin, cout))
        work = _f32((n,), dz.device)
        _lib.call("seis_unet_conv3x3_wgrad_ws", _lib.ptr(low), c1, _lib.ptr(skip),
                  skip.shape[-1], _lib.ptr(dz), N, H, W, cout, _lib.ptr(gw), _lib.ptr(gb),
                  _lib.ptr(work), _lib.stream_of(dz))

    def _flip_weights(self, like):
        """Weights of every layer's data gradient (all but the first layer's),
        in one launch: {name: (Cin, 9 * Cout)}."""
        layers = self.p.specs[1:]
        host = torch.tensor([[self.p.off[name][0], cout, cin] for name, cin, cout in layers],
                            dtype=torch.int64)
        sizes = [cout * 9 * cin for _, cin, cout in layers]
        wt = _bf((sum(sizes),), like.device)
        _lib.call("seis_unet_flip_layers", _lib.ptr(self.p.bf16), len(layers), _lib.ptr(host),
                  _lib.ptr(wt), _lib.stream_of(like))
        return {name: w for (name, _, _), w in zip(layers, wt.split(sizes))}

    def _dgrad(self, name, dz):
        """FP32 gradient of the layer's input."""
        _, cin, cout = next(s for s in self.p.specs if s[0] == name)
        _, _, (N, H, W) = self.saved[name]
        wt = self.wt[name]
        dx = _f32((N, H, W, cin), dz.device)
        _lib.call("seis_unet_conv3x3", _lib.ptr(dz), N, H, W, cout, _lib.ptr(wt), None, cin, 0,
                  None, None, _lib.ptr(dx), _lib.stream_of(dz))
        return dx

    def _dgrad_act(self, name, dz, before):
        """bf16 gradient of the pre-activation of layer `before`, whose output
        is this layer's input."""
        _, cin, cout = next(s for s in self.p.specs if s[0] == name)
        _, _, (N, H, W) = self.saved[name]
        z = self.saved[before][1]
        wt = self.wt[name]
        out = torch.empty_like(z)
        _lib.call("seis_unet_conv3x3_gelu_grad", _lib.ptr(dz), N, H, W, cout, _lib.ptr(wt), cin,
                  _lib.ptr(z), _lib.ptr(out), _lib.stream_of(dz))
        return out

    def _pair_bwd(self, level, dz, grad_arena, need_dx):
        """The two convolutions of a level (dz: gradient of the second's
        pre-activation); returns the FP32 gradient of the level's input."""
        self._wgrad(level + "b", dz, grad_arena)
        dz = self._dgrad_act(level + "b", dz, level + "a")
        self._wgrad(level + "a", dz, grad_arena)
        return self._dgrad(level + "a", dz) if need_dx else None

    def backward(self, dout, grad_arena):
        """dout (N, H, W) FP32 -> parameter gradients added into grad_arena
        (same layout as the master arena; the caller zeroes it)."""
        N, H, W = self.saved["shape"]
        s = _lib.stream_of(dout)
        C = self.p.base
        xh = self.saved["head_in"]
        hw, _ = self.p.head()
        gw, gb = self.p.head(grad_arena)
        dout = dout.contiguous()
        self.wt = self._flip_weights(dout)
        dz = torch.empty_like(xh)
        z = self.saved["dec0b"][1]
        if C == 32:
            _lib.call("seis_unet_head_gelu_bwd", _lib.ptr(xh), _lib.ptr(dout), N * H * W,
                      _lib.ptr(hw), _lib.ptr(z), _lib.ptr(dz), _lib.ptr(gw), _lib.ptr(gb), s)
        else:
            dx = _f32((N, H, W, C), dout.device)
            _lib.call("seis_unet_head_bwd", _lib.ptr(xh), _lib.ptr(dout), N * H * W, C,
                      _lib.ptr(hw), _lib.ptr(dx), _lib.ptr(gw), _lib.ptr(gb), s)
            _lib.call("seis_unet_gelu_bwd", _lib.ptr(dx), _lib.ptr(z), dx.numel(), _lib.ptr(dz),
                      s)
        # decoder, finest level first; the gradient of a concatenation's low
        # part goes on through the activation that made it, the skip's part is
        # read again by the encoder
        below = ("dec1b", "dec2b", "dec3b", "botb")
        cats = [None] * 4
        for l in (0, 1, 2, 3):
            cats[l] = self._pair_bwd(f"dec{l}", dz, grad_arena, True)
            _, _, (_, h, w) = self.saved[f"dec{l}a"]
            c2 = self.saved["skip_c"][l]
            z = self.saved[below[l]][1]
            dz = torch.empty_like(z)
            _lib.call("seis_unet_up_gelu_bwd", _lib.ptr(cats[l]), N, h, w,
                      cats[l].shape[-1] - c2, c2, _lib.ptr(z), _lib.ptr(dz), s)
        dpool = self._pair_bwd("bot", dz, grad_arena, True)
        for l in (3, 2, 1, 0):
            # gradient of the encoder output: skip path + pooled path
            z = self.saved[f"enc{l}b"][1]
            _, h, w, c2 = z.shape
            dz = torch.empty_like(z)
            _lib.call("seis_unet_skip_gelu_bwd", _lib.ptr(cats[l]), _lib.ptr(dpool), N, h, w,
                      cats[l].shape[-1] - c2, c2, _lib.ptr(z), _lib.ptr(dz), s)
            cats[l] = None
            dpool = self._pair_bwd(f"enc{l}", dz, grad_arena, l > 0)
        self.saved, self.wt = {}, None


class AdamW:
    """torch.optim.AdamW semantics (decoupled weight decay) on the flat arena."""

    def __init__(self, params, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=1e-2):
        self.p = params
        self.lr, self.betas, self.eps, self.wd = lr, betas, eps, weight_decay
        self.m = torch.zeros_like(params.master)
        self.v = torch.zeros_like(params.master)
        self.t = 0

    def step(self, grad):
        self.t += 1
        # the bf16 arena is refreshed in the same pass
        _lib.call("seis_unet_adamw", _lib.ptr(self.p.master), _lib.ptr(grad), _lib.ptr(self.m),
                  _lib.ptr(self.v), self.p.n, self.lr, self.betas[0], self.betas[1], self.eps,
                  self.wd, self.t, _lib.ptr(self.p.bf16), _lib.stream_of(grad))


def mse(pred, target, mask=None):
    """(loss tensor (1,), dpred) of mean((mask*(pred-target))^2)."""
    loss = _f32((1,), pred.device)
    dpred = torch.empty_like(pred)
    n = pred.numel()
    count = float(mask.sum()) if mask is not None else float(n)
    _lib.call("seis_unet_mse", _lib.ptr(pred), _lib.ptr(target), _lib.ptr(mask), n,
              1.0 / max(count, 1.0), _lib.ptr(loss), _lib.ptr(dpred), _lib.stream_of(pred))
    return loss, dpred


def train_step(net, opt, grad, model, scales, target, mask=None):
    """One AdamW step of the network on a batch; returns the loss tensor."""
    pred = net.forward(grad, model, scales, keep=True)
    loss, dpred = mse(pred, target, mask)
    g = torch.empty_like(net.p.master)
    _lib.call("seis_unet_fill", _lib.ptr(g), g.numel(), 0.0, _lib.stream_of(g))
    net.backward(dpred, g)
    opt.step(g)
    return loss


def input_scales(grad, model, vref=3000.0, vspan=1500.0):
    """Per-image (gscale, mscale, mshift): gradient normalised by its max |g|,
    model mapped to (v - vref) / vspan."""
    gmax = grad.abs().flatten(1).amax(1).clamp_min(1e-30)
    N = grad.shape[0]
    sc = torch.empty((N, 3), device=grad.device, dtype=torch.float32)
    sc[:, 0] = 1.0 / gmax
    sc[:, 1] = 1.0 / vspan
    sc[:, 2] = vref
    return sc
