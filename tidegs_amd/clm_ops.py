"""Drop-in for ``clm_kernels.fused_ssim`` (``clm_kernels/__init__.py:23-61``).

``fused_ssim(img1, img2, padding="same", train=True)`` returns the mean SSIM
(11x11 Gaussian window, sigma 1.5, C1 = 0.01^2, C2 = 0.03^2) and is
differentiable w.r.t. ``img1``; used inside TideGS's training loss
(``strategies/base_engine.py:472-488``).
"""
from __future__ import annotations

import torch

from . import _native as N

allowed_padding = ["same", "valid"]


class FusedSSIMMap(torch.autograd.Function):
    @staticmethod
    def forward(ctx, C1, C2, img1, img2, padding="same", train=True):
        img1 = img1.contiguous()
        img2 = img2.contiguous()
        N.require_cuda(img1, img2, names=["img1", "img2"])
        B, CH, H, W = img1.shape
        ssim_map = torch.empty_like(img1)
        if train:
            d1, d2, d3 = (torch.empty_like(img1) for _ in range(3))
        else:
            d1 = d2 = d3 = None
        N.call("tgs_fused_ssim_fwd", B, CH, H, W, float(C1), float(C2), N.ptr(img1), N.ptr(img2),
               N.ptr(ssim_map), N.ptr(d1), N.ptr(d2), N.ptr(d3), N.stream_handle())
        if padding == "valid":
            ssim_map = ssim_map[:, :, 5:-5, 5:-5]
        ctx.save_for_backward(img1.detach(), img2, d1, d2, d3)
        ctx.C1, ctx.C2, ctx.padding = C1, C2, padding
        return ssim_map

    @staticmethod
    def backward(ctx, opt_grad):
        img1, img2, d1, d2, d3 = ctx.saved_tensors
        if d1 is None:
            raise RuntimeError("fused_ssim backward needs train=True in the forward")
        dL_dmap = opt_grad
        if ctx.padding == "valid":
            dL_dmap = torch.zeros_like(img1)
            dL_dmap[:, :, 5:-5, 5:-5] = opt_grad
        dL_dmap = dL_dmap.contiguous()
        B, CH, H, W = img1.shape
        grad = torch.empty_like(img1)
        N.call("tgs_fused_ssim_bwd", B, CH, H, W, float(ctx.C1), float(ctx.C2), N.ptr(img1),
               N.ptr(img2), N.ptr(dL_dmap), N.ptr(d1), N.ptr(d2), N.ptr(d3), N.ptr(grad),
               N.stream_handle())
        return None, None, grad, None, None, None


class _FusedSSIMMean(torch.autograd.Function):
    """Mean SSIM in one forward launch (plus the sum of its partial sums) and
    one backward launch: neither the map nor the mean's constant gradient map
    is materialised.  A channels-last ``img1`` (a rendered [B,H,W,C] image seen
    as [B,C,H,W]) is read in place and its gradient comes back in its layout."""

    @staticmethod
    def forward(ctx, C1, C2, img1, img2, crop, train):
        channels_last = not img1.is_contiguous() and img1.permute(0, 2, 3, 1).is_contiguous()
        if not channels_last:
            img1 = img1.contiguous()
        img2 = img2.contiguous()
        N.require_cuda(img1.permute(0, 2, 3, 1) if channels_last else img1, img2,
                       names=["img1", "img2"])
        B, CH, H, W = img1.shape
        dev = img1.device
        keep = train and ctx.needs_input_grad[2]
        d1 = d2 = d3 = copy = None
        if keep:
            d1, d2, d3 = torch.empty((3, B, CH, H, W), dtype=torch.float32, device=dev)
            if channels_last:
                copy = torch.empty((B, CH, H, W), dtype=torch.float32, device=dev)
        partials = torch.empty(N.load().tgs_fused_ssim_mean_partials(B, CH, H, W),
                               dtype=torch.float64, device=dev)
        mean = torch.empty((), dtype=torch.float32, device=dev)
        N.call("tgs_fused_ssim_mean_fwd", B, CH, H, W, float(C1), float(C2), N.ptr(img1),
               int(channels_last), N.ptr(img2), crop, N.ptr(partials), N.ptr(mean), N.ptr(copy),
               N.ptr(d1), N.ptr(d2), N.ptr(d3), N.stream_handle())
        ctx.save_for_backward(copy if channels_last else img1.detach(), img2, d1, d2, d3)
        ctx.crop, ctx.train, ctx.channels_last = crop, train, channels_last
        return mean

    @staticmethod
    def backward(ctx, g):
        img1, img2, d1, d2, d3 = ctx.saved_tensors
        if not ctx.train:
            raise RuntimeError("fused_ssim backward needs train=True in the forward")
        if not ctx.needs_input_grad[2]:
            return None, None, None, None, None, None
        B, CH, H, W = img1.shape
        if ctx.channels_last:
            grad = torch.empty((B, H, W, CH), dtype=torch.float32,
                               device=img1.device).permute(0, 3, 1, 2)
        else:
            grad = torch.empty_like(img1)
        g = g.contiguous()
        N.call("tgs_fused_ssim_mean_bwd", B, CH, H, W, N.ptr(img1), N.ptr(img2), N.ptr(g),
               ctx.crop, N.ptr(d1), N.ptr(d2), N.ptr(d3), N.ptr(grad), int(ctx.channels_last),
               N.stream_handle())
        return None, None, grad, None, None, None


def fused_ssim(img1, img2, padding="same", train=True):
    C1 = 0.01 ** 2
    C2 = 0.03 ** 2
    assert padding in allowed_padding
    crop = 5 if padding == "valid" else 0
    B, CH, H, W = img1.shape
    if min(B, CH, H - 2 * crop, W - 2 * crop) <= 0:  # the mean of an empty map
        return FusedSSIMMap.apply(C1, C2, img1, img2, padding, train).mean()
    return _FusedSSIMMean.apply(C1, C2, img1, img2, crop, train)
