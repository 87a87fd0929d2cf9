"""Expert MLP with LoRA on gate/up/down as ONE autograd function
(reference: qwen3_moe_fused/kernels/fast_lora.py).

Shapes (rows B, hidden H, intermediate M, rank r, experts E):
    x (B,H);  G,U (E,M,H);  W (E,H,M);  Ag,Au (E,r,H);  Bg,Bu (E,M,r);  Aw (E,r,M);  Bw (E,H,r)
    e = G x + Sg Bg (Ag x),  g = U x + Su Bu (Au x),  h = silu(e) g,  y = W h + Sw Bw (Aw h)
Only e, g and the three rank-r activations Sg Ag x, Su Au x, Sw Aw h are kept for the backward pass.

Gradients.  With t = dOut Bproj (rows x r) and u = In Aproj^T (rows x r) for a projection
Out = (Wp + S Bp Ap) In:
    dAp = S t^T In        dBp = S dOut^T u        dIn = dOut Wp + S t Ap
Every LoRA gradient is therefore a rank-r grouped GEMM; the full (E, out, in) weight gradient
that the reference forms and then contracts (fast_lora.py:139-149) is never built.  Base weights
may be NF4 (``*qs`` not None): the forward and the input-gradient products decode them inside
the GEMM (the reference dequantises, fast_lora.py:57-62 "TODO: Fuse dequant and linear").
"""
from __future__ import annotations

from typing import List, Optional, Sequence, Tuple

import torch

from .. import _lib
from ..grouped_gemm.backward_dw import grouped_gemm_backward_dw as _dw
from ..grouped_gemm.forward import grouped_gemm_forward as _fwd
from ..grouped_gemm.forward_4bit import grouped_gemm_forward_4bit as _fwd4
from ..grouped_gemm.forward_4bit import grouped_gemm_forward_transposed_4bit as _dx4
from ..grouped_gemm.forward_transposed import grouped_gemm_forward_transposed as _dx
from ..grouped_gemm.fused import grouped_gemm_forward_4bit_lora as _fwd4_lora
from ..grouped_gemm.fused import grouped_gemm_forward_lora as _fwd_lora
from ..grouped_gemm.fused import grouped_glu_forward_4bit_lora as _glu4_lora
from ..grouped_gemm.fused import grouped_glu_forward_lora as _glu_lora
from ..grouped_gemm.fused import grouped_gemm_forward_transposed_4bit_dual_lora as _dx4_dual_lora
from ..grouped_gemm.fused import grouped_gemm_forward_transposed_4bit_lora as _dx4_lora
from ..grouped_gemm.fused import grouped_gemm_forward_transposed_lora as _dx_lora
from ..quantize.nf4 import dequantize_nf4, write_out_scales
from .silu_mul import silu_mul_backward_inplace, silu_mul_forward


def _packed_pair(x, Gqs, Uqs):
    """Whether the gate and up projections are packed matrices that one kernel takes for rows like ``x``."""
    return (Gqs is not None and Uqs is not None and x.dtype == torch.bfloat16 and x.shape[1] % 8 == 0
            and int(Gqs.blocksize) >= 8 and int(Uqs.blocksize) >= 8 and tuple(Gqs.shape) == tuple(Uqs.shape))


def _base_fwd(x, wq, wqs, m_sizes):
    if wqs is None:
        return _fwd(x, wq.to(x.dtype), m_sizes)
    if x.dtype == torch.bfloat16 and x.shape[1] % 8 == 0 and int(wqs.blocksize) >= 8:
        return _fwd4(x, wq, wqs, m_sizes)
    return _fwd(x, dequantize_nf4(wq, wqs, x.dtype), m_sizes)


def _dense(wq, wqs, dtype):
    return wq.to(dtype) if wqs is None else dequantize_nf4(wq, wqs, dtype)


def _proj_fwd(x, wq, wqs, a, b, s, m_sizes, us=None):
    """y = x W^T + (s x A^T) B^T; returns y and the scaled rank-r activation s x A^T (rows x r)."""
    if us is None:
        us = _fwd(x, a, m_sizes, alpha=s)
    if wqs is None and x.dtype == torch.bfloat16:
        # bf16 weights: the rank-r term rides in the reduction of the base product (no second pass over y)
        return _fwd_lora(x, wq.to(x.dtype), us, b, m_sizes), us
    if wqs is not None and x.dtype == torch.bfloat16 and x.shape[1] % 8 == 0 and int(wqs.blocksize) >= 8:
        return _fwd4_lora(x, wq, wqs, us, b, m_sizes), us   # the same over packed NF4 weights
    y = _base_fwd(x, wq, wqs, m_sizes)
    _fwd(us, b, m_sizes, out=y, accumulate=True)             # y += us b^T
    return y, us


def _proj_bwd_input(dout, ts, wq, wqs, a, m_sizes, out=None):
    """dIn (+)= dOut W + ts A with ts = s dOut B (rows x r)."""
    if wqs is None and dout.dtype == torch.bfloat16 and out is None:
        return _dx_lora(dout, wq.to(dout.dtype), ts, a, m_sizes)
    if wqs is not None and dout.dtype == torch.bfloat16 and out is None:
        return _dx4_lora(dout, wq, wqs, ts, a, m_sizes)
    if wqs is not None and dout.dtype == torch.bfloat16:
        out = _dx4(dout, wq, wqs, m_sizes, out=out, accumulate=out is not None)
    else:
        out = _dx(dout, _dense(wq, wqs, dout.dtype), m_sizes, out=out, accumulate=out is not None)
    return _dx(ts, a, m_sizes, out=out, accumulate=True)


# ---- joining and splitting the two adapters' thin matrices: all copies of a place in one launch
#
# A piece is (wide, narrow, dim, first, size): ``narrow`` (None: zeros) is ``wide``'s part of ``size`` from ``first`` on along
# ``dim``; a list of them is copied in the given direction.  One launch for what are three to four concatenations, fills
# and copies of the stock library; rank 16, 128 experts, a step's forward and backward: 72 -> 42 us at 65536 rows (137 MB),
# 51 -> 33 at 16384.
_Piece = Tuple[torch.Tensor, Optional[torch.Tensor], int, int, int]


def _copy_pieces(pieces: Sequence[_Piece], join: bool) -> None:
    jobs: List[_lib.BlockCopy] = []
    for wide, narrow, dim, first, size in pieces:
        es = wide.element_size()
        tail = es
        for n in wide.shape[dim + 1:]:
            tail *= n
        stride = wide.shape[dim] * tail
        blocks = wide.numel() * es // stride if stride else 0
        part = wide.data_ptr() + first * tail
        here = None if narrow is None else narrow.data_ptr()
        jobs.append(_lib.BlockCopy(here, part, blocks, size * tail, size * tail, stride) if join
                    else _lib.BlockCopy(part, here, blocks, size * tail, stride, size * tail))
    if jobs:
        rc = _lib.lib().mfl_copy_blocks((_lib.BlockCopy * len(jobs))(*jobs), len(jobs), _lib.stream())
        if rc == -6:  # MFL_ERR_UNSUPPORTED: runs that are no multiple of 16 bytes
            for wide, narrow, dim, first, size in pieces:
                part = wide.narrow(dim, first, size)
                if not join:
                    narrow.copy_(part)
                elif narrow is None:
                    part.zero_()
                else:
                    part.copy_(narrow)
            return
        _lib.check(rc, "mfl_copy_blocks")


def _joined(a: torch.Tensor, b: torch.Tensor, dim: int, pieces: List[_Piece]) -> torch.Tensor:
    """Room for ``torch.cat((a, b), dim)``; what fills it is added to ``pieces``."""
    dtype = torch.promote_types(a.dtype, b.dtype)  # (any strides and types, as the concatenation takes them)
    a, b = a.to(dtype).contiguous(), b.to(dtype).contiguous()
    assert a.shape[:dim] == b.shape[:dim] and a.shape[dim + 1:] == b.shape[dim + 1:]
    shape = list(a.shape)
    na, nb = a.shape[dim], b.shape[dim]
    shape[dim] = na + nb
    wide = torch.empty(shape, device=a.device, dtype=a.dtype)
    pieces += [(wide, a, dim, 0, na), (wide, b, dim, na, nb)]
    return wide


def _padded(b: torch.Tensor, dim: int, first: int, total: int, pieces: List[_Piece]) -> torch.Tensor:
    """Room for ``b`` in the columns from ``first`` on of ``total``, zeros in the others (one side of it)."""
    b = b.contiguous()
    size = b.shape[dim]
    assert 0 <= first <= total - size
    shape = list(b.shape)
    shape[dim] = total
    wide = torch.empty(shape, device=b.device, dtype=b.dtype)
    pieces += [(wide, b, dim, first, size), (wide, None, dim, 0 if first else size, total - size)]
    return wide


def _halves(wide: torch.Tensor, dim: int, size: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """``wide[..., :size, ...]`` and the rest along ``dim``, as tensors of their own."""
    assert wide.is_contiguous()
    out = []
    for n in (size, wide.shape[dim] - size):
        shape = list(wide.shape)
        shape[dim] = n
        out.append(torch.empty(shape, device=wide.device, dtype=wide.dtype))
    _copy_pieces([(wide, out[0], dim, 0, size), (wide, out[1], dim, size, wide.shape[dim] - size)], False)
    return out[0], out[1]


# from this many rows on, two thin products that stream the same wide operand are run as one of twice the rank
_WIDE_ROWS = 4096


class FastLora(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, Gq, Gqs, Ag, Bg, Sg, Uq, Uqs, Au, Bu, Su, Wq, Wqs, Aw, Bw, Sw, m_sizes):
        dt = x.dtype
        x = x.contiguous()
        Ag, Bg, Au, Bu, Aw, Bw = (p.to(dt).contiguous() for p in (Ag, Bg, Au, Bu, Aw, Bw))
        frozen_states = (Gqs, Uqs, Wqs)
        Gqs, Uqs, Wqs = write_out_scales(x, Gqs, Uqs, Wqs)
        ug = uu = ucat = None
        if Sg == Su and Ag.shape == Au.shape and x.shape[0] >= _WIDE_ROWS:
            # one pass over x for both adapters' rank-r activations
            r = Ag.shape[1]
            assert x.is_cuda and all(t.device == x.device for t in (Ag, Bg, Au, Bu))  # (the copies come before the products)
            pieces = []
            acat = _joined(Ag, Au, 1, pieces)
            # (hidden sizes in whole reduction steps of 64; others run the products by themselves, which then had a thin term of
            # twice the rank each: 8 experts, 384 x 672, 4788 rows 60 -> 71 us)
            packed = _packed_pair(x, Gqs, Uqs) and x.shape[1] % 64 == 0
            one_launch = Bg.shape == Bu.shape and (packed or (Gqs is None and Uqs is None and dt == torch.bfloat16
                                                              and Gq.dtype == dt and Uq.dtype == dt))
            if one_launch:
                # each matrix's thin weights are its adapter's B over its own columns of ucat and zeros over the other's (an
                # infinite activation of one adapter, whose row is not finite anyway, makes the other's product NaN there)
                assert Bg.shape[2] == r, "an adapter's A and B have one rank"
                bg, bu = _padded(Bg, 2, 0, 2 * r, pieces), _padded(Bu, 2, r, 2 * r, pieces)
            _copy_pieces(pieces, True)
            ucat = _fwd(x, acat, m_sizes, alpha=Sg)
            ug, uu = _halves(ucat, 1, r)
        if ucat is not None and one_launch:
            # gate, up, both rank-r terms and the SiLU-mul in one launch
            if packed:
                h, e, g = _glu4_lora(x, Gq, Gqs, Uq, Uqs, ucat, bg, bu, m_sizes)
            else:
                h, e, g = _glu_lora(x, Gq, Uq, ucat, bg, bu, m_sizes)
        else:
            e, ug = _proj_fwd(x, Gq, Gqs, Ag, Bg, Sg, m_sizes, ug)
            g, uu = _proj_fwd(x, Uq, Uqs, Au, Bu, Su, m_sizes, uu)
            h = silu_mul_forward(e, g)
        y, uw = _proj_fwd(h, Wq, Wqs, Aw, Bw, Sw, m_sizes)
        Gqs, Uqs, Wqs = frozen_states  # (the scales are written out again: 4 E N K / blocksize bytes each, 12.6 MB at 128 x 768 x 2048, not held between the passes)
        ctx.frozen = (Gq, Gqs, Sg, Uq, Uqs, Su, Wq, Wqs, Sw, m_sizes)
        ctx.save_for_backward(x, Ag, Bg, Au, Bu, Aw, Bw, e, g, ug, uu, uw)
        return y

    @staticmethod
    def backward(ctx, dy):
        Gq, Gqs, Sg, Uq, Uqs, Su, Wq, Wqs, Sw, m_sizes = ctx.frozen
        x, Ag, Bg, Au, Bu, Aw, Bw, e, g, ug, uu, uw = ctx.saved_tensors
        dt = x.dtype
        dy = dy.contiguous()
        if ctx.needs_input_grad[0]:
            Gqs, Uqs, Wqs = write_out_scales(dy, Gqs, Uqs, Wqs)

        # The rank-r activations carry the adapter's scaling (ug, uu, uw from the forward pass; tw, tu, tg here),
        # so every product below takes them as they are.
        # down projection
        tw = _dx(dy, Bw, m_sizes, alpha=Sw)                            # Sw dy Bw, rows x r
        dh = _proj_bwd_input(dy, tw, Wq, Wqs, Aw, m_sizes)
        silu_mul_backward_inplace(dh, e, g)                            # (dh, e, g) <- (h, de, dg)
        h, de, dg = dh, e, g
        dAw = _dw(h, tw, m_sizes, dt)                                  # (E, r, M)
        dBw = _dw(uw, dy, m_sizes, dt)                                 # (E, H, r)

        # up and gate projections
        tu = _dx(dg, Bu, m_sizes, alpha=Su)
        tg = _dx(de, Bg, m_sizes, alpha=Sg)
        pieces = []
        tcat = _joined(tg, tu, 1, pieces)
        acat = _joined(Ag, Au, 1, pieces) if ctx.needs_input_grad[0] else None
        _copy_pieces(pieces, True)
        if tg.shape == tu.shape and x.shape[0] >= _WIDE_ROWS and 2 * tg.shape[1] <= 64:
            # one pass over x for both: (E, 2 r, H)
            r = tg.shape[1]
            dAcat = _dw(x, tcat, m_sizes, dt)
            dAg, dAu = _halves(dAcat, 1, r)  # gradients of their own, not views
        else:
            dAu = _dw(x, tu, m_sizes, dt)                              # (E, r, H)
            dAg = _dw(x, tg, m_sizes, dt)
        dBu = _dw(uu, dg, m_sizes, dt)                                 # (E, M, r)
        dBg = _dw(ug, de, m_sizes, dt)

        dx = None
        if ctx.needs_input_grad[0]:
            if Gqs is None and Uqs is None and dt == torch.bfloat16 and Gq.dtype == dt and Uq.dtype == dt:
                # both base terms and both rank-r terms (side by side as one term of rank 2 r) in one reduction
                dx = _dx_lora(de, Gq, tcat, acat, m_sizes, dy2=dg, w2=Uq)
            elif _packed_pair(de, Gqs, Uqs):
                dx = _dx4_dual_lora(de, Gq, Gqs, dg, Uq, Uqs, tcat, acat, m_sizes)
            else:
                # both rank-r terms with the first base product, the second base product accumulates
                dx = _proj_bwd_input(de, tcat, Gq, Gqs, acat, m_sizes)
                if Uqs is not None and dt == torch.bfloat16:
                    _dx4(dg, Uq, Uqs, m_sizes, out=dx, accumulate=True)
                else:
                    _dx(dg, _dense(Uq, Uqs, dt), m_sizes, out=dx, accumulate=True)

        return (dx, None, None, dAg, dBg, None, None, None, dAu, dBu, None, None, None, dAw, dBw, None, None)


fast_lora = FastLora.apply
