"""Truncated 2-D DFTs for the spectral layer.

Sp_SpectralConv2D keeps only the modes kh in [0, m) and [r-m, r), kw in [0, m) of rfft2(x) and feeds
irfft2 a spectrum that is zero everywhere else (reference: network/sp_layer.py:138-150).  Computing
exactly those modes as two small matrix products per direction,

    forward   Y[n,h,c,kw]  = sum_w x[n,h,w,c] e^{-2 pi i kw w / r} / sqrt(r)
              Z[n,kh,c,kw] = sum_h Y[n,h,c,kw] e^{-2 pi i kh h / r} / sqrt(r)
    inverse   U[n,h,o,kw]  = sum_kh O[n,kh,o,kw] e^{+2 pi i kh h / r} / sqrt(r)
              y[n,h,w,o]   = Re sum_kw c_kw U[n,h,o,kw] e^{+2 pi i kw w / r} / sqrt(r),   c_0 = 1, c_kw = 2
                             (c = 1 as well for the Nyquist column of an even r),

gives the same result as the FFT route up to fp32 rounding (the real part in the last line is what the
complex-to-real transform of irfft2 computes from a half spectrum), works directly on the [N, r, r, C]
layout of the module - both full-tensor transposes, the full-size spectra, the corner gather/scatter and
the zero fill disappear - and does not depend on r having small prime factors (r = 211 is prime).
The two products along w, which touch the full tensor, are the HIP kernels behind `truncated_dft_rows_*`;
the two small ones along h are library GEMMs; the per-mode channel contraction between them is the HIP
kernel behind `spectral_modes_compact`.
"""
import math
from typing import Dict, NamedTuple, Tuple

import torch
from torch import Tensor

from ..extension.bind.linear import _aligned, linear_weight_grad
from ..extension.bind.datamove import (_spectral_linear_backward_supported, _spectral_linear_input_grad_into,
                                       _spectral_weight_adjoint, _spectral_weight_grad, inverse_table_operand, keep_padded,
                                       pad_dft_table, spectral_inverse_linear, spectral_inverse_linear_supported,
                                       spectral_modes_compact, spectral_modes_middle, spectral_modes_middle_supported,
                                       truncated_dft_rows_forward, truncated_dft_rows_inverse, truncated_dft_rows_supported)


class _Tables(NamedTuple):
    forms: Tuple[Tensor, Tensor, Tensor, Tensor]  # Fw, Gh, Ghi, Fwi
    operand: Tensor                               # operand table of Fwi: the layer's last kernel
    adjoint: Tuple[Tensor, Tensor, Tensor]        # conj(Ghi)^T, conj(Gh)^T, operand table of Fw: the backward


_TABLES: Dict[Tuple[int, int, str], _Tables] = {}


def _tables(r: int, m: int, device) -> _Tables:
    """Everything that the layer keeps for a size, for both directions: formed on the host in fp64 and copied over, which
    waits for the copy, so that any stream may read it at once and no captured graph owns it."""
    key = (r, m, str(device))
    if key not in _TABLES:
        with torch.inference_mode(False), torch.no_grad():
            idx = torch.arange(r, dtype=torch.float64, device="cpu")
            kw = torch.arange(m, dtype=torch.float64, device="cpu")
            kh = torch.cat([kw, kw + (r - m)])
            s = 1.0 / math.sqrt(r)
            ang_w = 2.0 * math.pi * idx[:, None] * kw[None, :] / r                  # [r, m]
            fw = torch.stack([torch.cos(ang_w), -torch.sin(ang_w)], dim=-1) * s      # columns (kw, re|im)
            c = torch.full((m,), 2.0, dtype=torch.float64, device="cpu")
            c[0] = 1.0
            if r % 2 == 0 and m - 1 == r // 2:
                c[-1] = 1.0
            fwi = torch.stack([torch.cos(ang_w) * c, -torch.sin(ang_w) * c], dim=-1) * s
            ang_h = 2.0 * math.pi * kh[:, None] * idx[None, :] / r                  # [2m, r]
            gh = (torch.complex(torch.cos(ang_h), -torch.sin(ang_h)) * s).to(torch.complex64)
            ghi = (torch.complex(torch.cos(ang_h), torch.sin(ang_h)).t() * s).to(torch.complex64).contiguous()
            fw, fwi = fw.reshape(r, 2 * m).float(), fwi.reshape(r, 2 * m).float()
            upload = lambda *tables: tuple(t.to(device) for t in tables)
            forms = upload(fw, gh, ghi, fwi)
            if 2 * m <= 64:  # the row kernels' own forms
                for table, host in ((forms[0], fw), (forms[3], fwi)):
                    keep_padded(table, *upload(pad_dft_table(host, False), pad_dft_table(host, True)))
                operand, = upload(inverse_table_operand(fwi))
                adjoint = upload(ghi.t().conj().resolve_conj().contiguous(), gh.t().conj().resolve_conj().contiguous(),
                                 inverse_table_operand(fw))
            else:
                operand = adjoint = None  # no kernel takes as many modes
            _TABLES[key] = _Tables(forms, operand, adjoint)
    return _TABLES[key]


def dft_tables(r: int, m: int, device) -> Tuple[Tensor, Tensor, Tensor, Tensor]:
    """(Fw [r, 2m] real, Gh [2m, r] complex, Ghi [r, 2m] complex, Fwi [r, 2m] real), built in fp64."""
    return _tables(r, m, device).forms


def _operand_table(r: int, m: int, device) -> Tensor:
    return _tables(r, m, device).operand


def _adjoint_tables(r: int, m: int, device):
    """(conj(Ghi)^T [2m, r], conj(Gh)^T [r, 2m], operand table of Fw): what the backward of the layer's linear part takes."""
    return _tables(r, m, device).adjoint


def supported(r: int, m: int) -> bool:
    """The two retained row windows must not overlap."""
    return 2 * m <= r


def fused_tail_supported(r: int, cin: int, cout: int, m: int) -> bool:
    """True when spectral_modes_apply_linear runs in three launches (row DFT, retained modes, inverse row DFT fused
    with the residual Linear and the activation)."""
    return (truncated_dft_rows_supported(r, cin, m) and spectral_modes_middle_supported(r, cin, cout, m) and
            spectral_inverse_linear_supported(r, cin, cout, m))


def spectral_modes_apply_linear(x: Tensor, weight_1: Tensor, weight_2: Tensor, m: int, linear_weight_kn: Tensor,
                                linear_bias, activation) -> Tensor:
    """act(x @ linear_weight_kn + linear_bias + irfft2(W . truncate(rfft2(x)))) for x [N, r, r, C]: the whole
    spectral layer after dropout; requires fused_tail_supported."""
    N, r, _, cin = x.shape
    fw, gh, ghi, fwi = dft_tables(r, m, x.device)
    yp = truncated_dft_rows_forward(x, fw, planar=True)             # [N, 2m, r, Cin]
    up = spectral_modes_middle(yp, gh, ghi, weight_1, weight_2)     # [N, 2m, r, Cout]
    return spectral_inverse_linear(up, _operand_table(r, m, x.device), x, linear_weight_kn, linear_bias, activation)


class _DifferentiatedOnce(torch.autograd.Function):
    """_DifferentiatedOnce.apply(n, *gradients, *sources): the n gradients, as functions of what they were formed from that
    cannot be differentiated.  (Without the sources, autograd would not find this node on its way to them and take the
    gradients for constants.)"""

    @staticmethod
    def forward(ctx, n, *tensors):
        return tuple(g.clone() for g in tensors[:n])  # (views may not be changed in place later)

    @staticmethod
    def backward(ctx, *grads):
        raise RuntimeError("the spectral layer's gradients cannot be differentiated: its training route (use_truncated_dft) "
                           "can be differentiated once, not twice")


class _SpectralLinearFunction(torch.autograd.Function):
    """x @ W_lin^T + b + irfft2(W_f . truncate(rfft2(x))) on the truncated-DFT route, with its backward on the same
    kernels.  Every stage is linear, so the backward runs the adjoint stages in reverse: the inverse row transform's
    adjoint is a forward row transform with the inverse table, the forward one's an inverse row transform with the
    forward table, and the adjoint of the complex-linear middle (DFT along h, channel contraction, inverse DFT
    along h) is the same kernel with conjugate-transposed tables and weights.  The Fourier weights' gradient,
    dW[kh, kw, c, o] = sum_n conj(Z[n, kh, c, kw]) dO[n, kh, o, kw], is formed from the retained modes (a few MB) by a
    DFT along h and outer products; the adjoint row transform and g @ W_lin are one kernel, as in the forward.
    The kernels record nothing: under create_graph the gradients come out such that a second derivative through any of
    them raises."""

    @staticmethod
    def forward(ctx, x, weight_1, weight_2, lin_weight, lin_bias, lin_weight_kn, m):
        N, r, _, cin = x.shape
        fw, gh, ghi, _ = dft_tables(r, m, x.device)
        yp = truncated_dft_rows_forward(x, fw, planar=True)                         # [N, 2m, r, Cin]
        up = spectral_modes_middle(yp, gh, ghi, weight_1, weight_2)                 # [N, 2m, r, Cout]
        out = spectral_inverse_linear(up, _operand_table(r, m, x.device), x, lin_weight_kn, lin_bias, None)
        ctx.save_for_backward(x, weight_1, weight_2, lin_weight, yp)
        ctx.m, ctx.has_bias = m, lin_bias is not None
        return out

    @staticmethod
    def backward(ctx, g):
        if not torch.is_grad_enabled():
            return _SpectralLinearFunction._gradients(ctx, g)
        with torch.no_grad():
            grads = _SpectralLinearFunction._gradients(ctx, g)
        formed = [t for t in grads if t is not None]
        once = iter(_DifferentiatedOnce.apply(len(formed), *formed, g, *ctx.saved_tensors[:4]))
        return tuple(None if t is None else next(once) for t in grads)

    @staticmethod
    def _gradients(ctx, g):
        x, weight_1, weight_2, lin_weight, yp = ctx.saved_tensors
        m = ctx.m
        g = _aligned(g.contiguous())
        r, cout = g.shape[1], g.shape[3]
        cin = x.shape[-1]
        _, gh, _, fwi = dft_tables(r, m, x.device)
        ghi_h, gh_h, fw_operand = _adjoint_tables(r, m, x.device)                   # [2m, r], [r, 2m]
        dup = truncated_dft_rows_forward(g, fwi, planar=True)                       # [N, 2m, r, Cout] = Fi^T g
        dx = None
        if ctx.needs_input_grad[0]:
            # the middle kernel writes at most 64 channels per call, and so does the adjoint of the layer's last kernel
            width = min(cin, 64)
            wh = _spectral_weight_adjoint(weight_1.detach().contiguous(), weight_2.detach().contiguous(), width)
            w = lin_weight.detach().contiguous()                                    # [Cout, Cin]
            dyp = [spectral_modes_middle(dup, ghi_h, gh_h, w1h, w2h) for w1h, w2h in wh]  # each [N, 2m, r, width]
            dx = torch.empty_like(x)
            for i, slice_ in enumerate(dyp):
                _spectral_linear_input_grad_into(dx, i * width, slice_, fw_operand, g, w)
        dw_lin = db = dw1 = dw2 = None
        if ctx.needs_input_grad[3] or (ctx.has_bias and ctx.needs_input_grad[4]):
            dw_lin, db = linear_weight_grad(x.view(-1, cin), g.view(-1, cout), out_major=True)
            if not ctx.has_bias:
                db = None
        if ctx.needs_input_grad[1] or ctx.needs_input_grad[2]:
            dw = _spectral_weight_grad(yp, gh, dup, ghi_h)                          # [2m, kw, Cin, Cout, 2]
            dw1, dw2 = dw[:m], dw[m:]
        return dx, dw1, dw2, dw_lin, db, None, None


def spectral_linear_trainable(r: int, cin: int, cout: int, m: int) -> bool:
    """True when spectral_linear_train serves this shape: the three-launch route forward, and for the backward a
    row-transform variant for both widths, kernels for its last stage and for the Fourier weights' gradient, and a
    weight-gradient row length that is a multiple of 4."""
    return (fused_tail_supported(r, cin, cout, m) and truncated_dft_rows_supported(r, cout, m) and
            spectral_modes_middle_supported(r, cout, min(cin, 64), m) and
            _spectral_linear_backward_supported(r, cin, cout, m) and cout % 4 == 0)


def spectral_linear_train(x: Tensor, weight_1: Tensor, weight_2: Tensor, m: int, lin_weight: Tensor, lin_bias,
                          lin_weight_kn: Tensor) -> Tensor:
    """x @ lin_weight^T + lin_bias + irfft2(W . truncate(rfft2(x))) for x [N, r, r, Cin], with an autograd graph
    (see _SpectralLinearFunction); requires spectral_linear_trainable."""
    return _SpectralLinearFunction.apply(x, weight_1, weight_2, lin_weight, lin_bias, lin_weight_kn, m)


def spectral_modes_apply(x: Tensor, weight_1: Tensor, weight_2: Tensor, m: int) -> Tensor:
    """x [N, r, r, Cin] -> irfft2(W . truncate(rfft2(x))) as [N, r, r, Cout] (norm='ortho')."""
    N, r, _, cin = x.shape
    cout = weight_1.shape[3]
    fw, gh, ghi, fwi = dft_tables(r, m, x.device)
    rows_kernel = truncated_dft_rows_supported(r, cin, m) and truncated_dft_rows_supported(r, cout, m)
    if rows_kernel and spectral_modes_middle_supported(r, cin, cout, m):
        # three launches: DFT along w, everything on the retained modes, inverse DFT along w
        yp = truncated_dft_rows_forward(x, fw, planar=True)                               # [N, 2m, r, Cin]
        up = spectral_modes_middle(yp, gh, ghi, weight_1, weight_2)                       # [N, 2m, r, Cout]
        return truncated_dft_rows_inverse(up, fwi, planar=True)                           # [N, r, r, Cout]
    if rows_kernel:
        y = truncated_dft_rows_forward(x.reshape(N * r, r, cin), fw)                     # [N r, Cin, 2m]
    else:
        y = torch.matmul(x.reshape(N * r, r, cin).transpose(1, 2), fw)
    yc = torch.view_as_complex(y.view(N, r, cin, m, 2)).reshape(N, r, cin * m)
    z = torch.matmul(gh, yc).view(N, 2 * m, cin, m)                                      # [N, 2m, Cin, m]
    o = spectral_modes_compact(z, weight_1, weight_2)                                    # [N, 2m, Cout, m]
    u = torch.matmul(ghi, o.view(N, 2 * m, cout * m))                                    # [N, r, Cout m]
    ur = torch.view_as_real(u).view(N * r, cout, 2 * m)
    if rows_kernel:
        return truncated_dft_rows_inverse(ur, fwi).view(N, r, r, cout)
    return torch.matmul(fwi, ur.transpose(1, 2)).view(N, r, r, cout)
