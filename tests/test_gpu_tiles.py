"""The tiles of the row-grouped bf16 products: which of them a product runs on, and the results at their borders.

The tests of the single products take small shapes, whose launches are spread over the smallest tiles; what is here has
enough tiles for the large ones, and asks the names of the launched kernels so that a later rule cannot take it elsewhere
unseen."""
import numpy as np
import pytest
import torch

import oracle
from util import check_close, check_tiles, gen, randn, to_np32

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.grouped_gemm.forward import grouped_gemm_forward  # noqa: E402
from qwen3_moe_fused.grouped_gemm.forward_4bit import (grouped_gemm_forward_4bit,  # noqa: E402
                                                       grouped_gemm_forward_transposed_4bit)
from qwen3_moe_fused.grouped_gemm.forward_transposed import grouped_gemm_forward_transposed  # noqa: E402
from qwen3_moe_fused.grouped_gemm.fused import (grouped_gemm_forward_4bit_gathered,  # noqa: E402
                                                grouped_gemm_forward_4bit_lora, grouped_gemm_forward_gathered,
                                                grouped_gemm_forward_lora, grouped_gemm_forward_transposed_4bit_lora,
                                                grouped_gemm_forward_transposed_dual, grouped_gemm_forward_transposed_lora,
                                                grouped_gemm_forward_transposed_silu_bwd, grouped_glu_forward,
                                                grouped_glu_forward_4bit, grouped_glu_forward_lora)
from qwen3_moe_fused.kernels.silu_mul import silu_mul_backward, silu_mul_forward  # noqa: E402
from qwen3_moe_fused.quantize.nf4 import Nf4QuantState, nf4_code  # noqa: E402

DEV = "cuda"
FWD, DX = 0, 1


# rows per expert, N, experts, square: the gated product's 256 x 256 tiles only where they need fewer rounds over the CUs.
# 64 experts, N = 832, K = 2208: 253 us on them against 211 on 320 x 192 at 304 rows; 128 experts, N = 768: 350 against 312
# at 300, 195 against 203 at 128, 409 against 447 at 400.
@pytest.mark.parametrize("rows,N,E,square", [(304, 832, 64, False), (300, 768, 128, False), (311, 448, 128, False),
                                             (128, 768, 128, True), (188, 768, 128, True), (400, 768, 128, True)])
def test_gated_product_takes_the_tiles_of_fewer_rounds(rows, N, E, square):
    R, K = rows * E, 64
    g = gen(R + N)
    ms = torch.full((E,), rows, dtype=torch.int32)
    ms[0], ms[1], ms[2] = 0, rows + 7, 2 * rows - 7
    x = randn((R, K), g, 1.0, torch.bfloat16)
    wg, wu = (randn((E, N, K), g, 0.05, torch.bfloat16) for _ in range(2))
    mb = 256 if square else 320
    h, e, gg = check_tiles(lambda: grouped_glu_forward(x.to(DEV), wg.to(DEV), wu.to(DEV), ms.to(DEV), return_products=True),
                           ("pipe", mb, 256 if square else 192, FWD, False, 1))
    rows_checked = np.r_[0:3 * rows, R - rows:R]  # the experts at the borders and the last one
    sel = oracle.sel_from_m_sizes(ms.numpy())[rows_checked]
    for out, w, what in ((e, wg, "gate"), (gg, wu, "up")):
        check_close(out[rows_checked], oracle.linear_fwd(to_np32(x[rows_checked]), to_np32(w), sel), what=what)
    assert torch.equal(h, silu_mul_forward(e, gg))


# Rows per expert at the borders of the tiles, experts without rows and of several tiles; the last column slice holds 8, 24 or
# 32 columns or is whole; reductions of one step and of odd and even numbers of them.
TALL = [319, 320, 321, 0, 1, 700, 290, 640, 33, 288] * 4       # 320 x 192
WIDE_OUT = [191, 192, 193, 0, 1, 150, 400, 97, 129, 32] * 4    # 192 x 256, where the kernel has it
WIDE_MID = [255, 256, 257, 0, 190, 520, 1, 180, 64, 300] * 4   # 256 x 256 below 512 rows per expert
SQUARE = [513, 255, 256, 257, 0, 1, 2047, 31, 700, 640, 512, 1100]
PAIR = [160, 161, 159, 0, 1, 320, 321, 1280]                   # 160 x 128, few experts

# shape -> m_sizes, N, K, then the tiles: (kernel, rows, columns) of the plain products, of those with a thin term, of those
# that only the pipelined kernel has (gathered rows, accumulated or float32 results, the gated unit's backward)
SHAPES = {
    "tall": (TALL, 584, 192, ("wide", 320, 192), ("wide", 320, 192), ("pipe", 320, 192)),
    "wide_out": (WIDE_OUT, 1024, 64, ("wide", 192, 256), ("wide", 320, 192), ("pipe", 320, 192)),
    "wide_mid": (WIDE_MID, 1024, 192, ("wide", 256, 256), ("wide", 256, 256), ("pipe", 320, 192)),
    "square": (SQUARE, 1288, 128, ("wide", 256, 256), ("wide", 256, 256), ("pipe", 256, 256)),
    "pair": (PAIR, 1912, 192, ("pipe", 160, 128), ("pipe", 160, 128), ("pipe", 160, 128)),
}


class Case:
    """Operands of the products of one shape, and their results by the oracle.  Input gradients take weights of (E, K, N), so
    that their outputs have the same N columns."""

    def __init__(self, m_sizes, N, K, r=16):
        E, R = len(m_sizes), sum(m_sizes)
        self.g = gen(R + N + K)
        rows, weight = lambda n: randn((R, n), self.g, 1.0, torch.bfloat16), lambda k: randn((E, N, k), self.g, 0.05, torch.bfloat16)
        host = {"x": rows(K), "x2": rows(K), "w": weight(K), "w2": weight(K), "u": rows(r), "b": weight(r), "b2": weight(r)}
        self.ms_host = torch.tensor(m_sizes, dtype=torch.int32)
        self.sel, self.R, self.E = oracle.sel_from_m_sizes(self.ms_host.numpy()), R, E
        product = lambda a, w: oracle.linear_fwd(to_np32(host[a]), to_np32(host[w]), self.sel).astype(np.float64)
        self.xw, self.xw2, self.x2w2, self.ub = product("x", "w"), product("x", "w2"), product("x2", "w2"), product("u", "b")
        self.ub2 = product("u", "b2")
        for name, t in host.items():
            setattr(self, name, t.to(DEV))
            if t.ndim == 3:
                setattr(self, name + "t", t.transpose(1, 2).contiguous().to(DEV))
        self.ms = self.ms_host.to(DEV)

    def gather(self, div=2):
        """(source, row indices): the rows of x from a source in which each appears once among others."""
        T = self.R // div + 5
        idx = torch.randperm(T * div, generator=self.g)[:self.R].to(torch.int32).to(DEV)
        src = randn((T, self.x.shape[1]), self.g, 1.0, torch.bfloat16).to(DEV)
        return src, idx, div


@pytest.mark.parametrize("shape", SHAPES)
def test_plain_and_two_term_products(shape):
    c, tile = Case(*SHAPES[shape][:3]), SHAPES[shape][3]
    y = check_tiles(lambda: grouped_gemm_forward(c.x, c.w, c.ms), (*tile, FWD, False, 0))
    check_close(y, c.xw, what="forward")
    dx = check_tiles(lambda: grouped_gemm_forward_transposed(c.x, c.wt, c.ms), (*tile, DX, False, 0))
    check_close(dx, c.xw, what="input gradient")
    both = check_tiles(lambda: grouped_gemm_forward_transposed_dual(c.x, c.wt, c.x2, c.w2t, c.ms), (*tile, DX, False, 0))
    check_close(both, c.xw + c.x2w2, what="input gradient, two terms")
    joined = grouped_gemm_forward_transposed(torch.cat([c.x, c.x2], 1), torch.cat([c.wt, c.w2t], 1).contiguous(), c.ms)
    assert torch.equal(both, joined), "the same reduction in the same order"


@pytest.mark.parametrize("shape", SHAPES)
def test_products_with_a_thin_term(shape):
    c, tile = Case(*SHAPES[shape][:3]), SHAPES[shape][4]
    y = check_tiles(lambda: grouped_gemm_forward_lora(c.x, c.w, c.u, c.b, c.ms), (*tile, FWD, False, 2))
    check_close(y, c.xw + c.ub, what="forward")
    joined = grouped_gemm_forward(torch.cat([c.x, c.u], 1), torch.cat([c.w, c.b], 2).contiguous(), c.ms)
    assert torch.equal(y, joined), "the same reduction in the same order"
    dx = check_tiles(lambda: grouped_gemm_forward_transposed_lora(c.x, c.wt, c.u, c.bt, c.ms), (*tile, DX, False, 2))
    check_close(dx, c.xw + c.ub, what="input gradient")
    both = check_tiles(lambda: grouped_gemm_forward_transposed_lora(c.x, c.wt, c.u, c.bt, c.ms, dy2=c.x2, w2=c.w2t),
                       (*tile, DX, False, 2))
    check_close(both, c.xw + c.x2w2 + c.ub, what="input gradient, two terms")
    joined = grouped_gemm_forward_transposed(torch.cat([c.x, c.x2, c.u], 1), torch.cat([c.wt, c.w2t, c.bt], 1).contiguous(),
                                             c.ms)
    assert torch.equal(both, joined), "the same reduction in the same order"
    tile = SHAPES[shape][5]
    y = check_tiles(lambda: grouped_gemm_forward_lora(c.x, c.w, c.u, c.b, c.ms, torch.float32), (*tile, FWD, False, 2))
    check_close(y, c.xw + c.ub, 1e-4, 1e-4, "forward, float32 result")
    dx = check_tiles(lambda: grouped_gemm_forward_transposed_lora(c.x, c.wt, c.u, c.bt, c.ms, torch.float32),
                     (*tile, DX, False, 2))
    check_close(dx, c.xw + c.ub, 1e-4, 1e-4, "input gradient, float32 result")


# Parts of 96 columns: a wave's store starts in the middle of a row (store 1 in row 5 at column 32, 2 in row 10 at 64, 4 in
# row 21 at 32, 5 in row 26 at 64).  Experts that end in just these rows, with 32 columns left to either wave, have stores
# without a lane; one that was counted all the same let the next tile's second step be read before it had landed.
@pytest.mark.parametrize("N", [224, 320])
def test_last_rows_in_which_a_store_has_no_lane(N):
    m_sizes = [54, 59, 38, 43, 70, 75, 22, 27, 86, 11, 6, 102] * 16
    c = Case(m_sizes, N, 384)
    tile = ("wide", 320, 192)
    products = {
        "forward": (lambda: grouped_gemm_forward(c.x, c.w, c.ms), c.xw, FWD, 0),
        "input gradient": (lambda: grouped_gemm_forward_transposed(c.x, c.wt, c.ms), c.xw, DX, 0),
        "forward, thin term": (lambda: grouped_gemm_forward_lora(c.x, c.w, c.u, c.b, c.ms), c.xw + c.ub, FWD, 2),
        "input gradient, two terms and the thin one":
            (lambda: grouped_gemm_forward_transposed_lora(c.x, c.wt, c.u, c.bt, c.ms, dy2=c.x2, w2=c.w2t),
             c.xw + c.x2w2 + c.ub, DX, 2),
    }
    for what, (product, expect, mode, fusion) in products.items():
        y = check_tiles(product, (*tile, mode, False, fusion))
        check_close(y, expect, what=what)
        for _ in range(20):
            assert torch.equal(product(), y), f"{what}: the same bits from run to run"


@pytest.mark.parametrize("shape", SHAPES)
def test_products_of_the_pipelined_kernel(shape):
    c, tile = Case(*SHAPES[shape][:3]), SHAPES[shape][5]
    src, idx, div = c.gather()
    rows = src[(idx // div).long()]
    y = check_tiles(lambda: grouped_gemm_forward_gathered(src, idx, div, c.w, c.ms), (*tile, FWD, False, 0))
    assert torch.equal(y, grouped_gemm_forward(rows.contiguous(), c.w, c.ms)), "gathered rows"
    for product, w, mode in ((grouped_gemm_forward, c.w, FWD), (grouped_gemm_forward_transposed, c.wt, DX)):
        y = check_tiles(lambda: product(c.x, w, c.ms, torch.float32), (*tile, mode, False, 0))
        check_close(y, c.xw, 1e-4, 1e-4, "float32 result")
        out = c.x2w2.astype(np.float32)
        out_dev = torch.from_numpy(out).to(DEV).bfloat16()
        start = to_np32(out_dev).astype(np.float64)
        check_tiles(lambda: product(c.x, w, c.ms, out=out_dev, alpha=0.5, accumulate=True), (*tile, mode, False, 0))
        check_close(out_dev, start + 0.5 * c.xw, what="accumulated")
    e, g = (randn(c.xw.shape, c.g, s, torch.bfloat16).to(DEV) for s in (2.0, 1.0))
    got = check_tiles(lambda: grouped_gemm_forward_transposed_silu_bwd(c.x, c.wt, e, g, c.ms, return_h=True),
                      (*tile, DX, False, 4))
    de, dg = silu_mul_backward(grouped_gemm_forward_transposed(c.x, c.wt, c.ms), e, g)
    for a, b, what in zip(got, (de, dg, silu_mul_forward(e, g)), ("de", "dg", "h")):
        assert torch.equal(a, b), f"{what}: the same bits as the product, then the gated unit's backward"


# K % 64 != 0: the last step is a partial one
@pytest.mark.parametrize("m_sizes,N,rows,columns", [(TALL, 584, 320, 192), (SQUARE, 1288, 256, 256), (PAIR, 1912, 160, 128)])
def test_reductions_that_end_inside_a_step(m_sizes, N, rows, columns):
    c = Case(m_sizes, N, 72)
    tile = ("pipe", rows, columns)
    check_close(check_tiles(lambda: grouped_gemm_forward(c.x, c.w, c.ms), (*tile, FWD, False, 0)), c.xw, what="forward")
    check_close(check_tiles(lambda: grouped_gemm_forward_transposed(c.x, c.wt, c.ms), (*tile, DX, False, 0)), c.xw,
                what="input gradient")
    check_close(check_tiles(lambda: grouped_gemm_forward_lora(c.x, c.w, c.u, c.b, c.ms), (*tile, FWD, False, 2)), c.xw + c.ub,
                what="forward, thin term")
    check_close(check_tiles(lambda: grouped_gemm_forward_transposed_lora(c.x, c.wt, c.u, c.bt, c.ms), (*tile, DX, False, 2)),
                c.xw + c.ub, what="input gradient, thin term")


# the gated product counts its tiles by its own rules: 128, 96 or 64 columns of each matrix in a tile
@pytest.mark.parametrize("m_sizes,N,K,rows,columns", [(TALL, 584, 192, 320, 192), (WIDE_MID, 760, 64, 256, 256),
                                                      (SQUARE, 1288, 128, 256, 256), (PAIR, 984, 192, 160, 128)])
def test_gated_products(m_sizes, N, K, rows, columns):
    c = Case(m_sizes, N, K)
    tile = ("pipe", rows, columns, FWD, False)
    h, e, g = check_tiles(lambda: grouped_glu_forward(c.x, c.w, c.w2, c.ms, return_products=True), (*tile, 1))
    check_close(e, c.xw, what="gate")
    check_close(g, c.xw2, what="up")
    assert torch.equal(h, silu_mul_forward(e, g))
    src, idx, div = c.gather()
    h = check_tiles(lambda: grouped_glu_forward(src, c.w, c.w2, c.ms, idx, div), (*tile, 1))
    x = src[(idx // div).long()].contiguous()
    assert torch.equal(h, silu_mul_forward(grouped_gemm_forward(x, c.w, c.ms), grouped_gemm_forward(x, c.w2, c.ms)))
    h, e, g = check_tiles(lambda: grouped_glu_forward_lora(c.x, c.w, c.w2, c.u, c.b, c.b2, c.ms), (*tile, 3))
    check_close(e, c.xw + c.ub, what="gate, thin term")
    check_close(g, c.xw2 + c.ub2, what="up, thin term")
    assert torch.equal(h, silu_mul_forward(e, g))


class Packed(Case):
    """The same with NF4 weights: w and w2 (E, N, K) for the forward products, wt (E, K, N) for the input gradient."""

    def __init__(self, m_sizes, N, K, blocksize):
        super().__init__(m_sizes, N, K)
        for name in ("w", "w2", "wt"):
            q, absmax = oracle.nf4_quant(to_np32(getattr(self, name)), blocksize)
            shape = getattr(self, name).shape
            setattr(self, name + "_deq", oracle.round_bf16(oracle.nf4_dequant(q, absmax, blocksize)).reshape(shape))
            state = Nf4QuantState(absmax=torch.from_numpy(absmax).to(DEV), shape=tuple(shape), code=nf4_code(DEV),
                                  blocksize=blocksize, dtype=torch.bfloat16)
            setattr(self, name + "_q", (torch.from_numpy(q).view(-1, 1).to(DEV), state))
        x = to_np32(self.x)
        self.xw = oracle.linear_fwd(x, self.w_deq, self.sel).astype(np.float64)
        self.xw2 = oracle.linear_fwd(x, self.w2_deq, self.sel).astype(np.float64)
        self.dx = oracle.linear_bwd_input(x, self.wt_deq, self.sel).astype(np.float64)


# N, K, block size, rows and columns of the tiles; K % 128 != 0: the streaming kernel, which takes the plain and the gated
# forward product of few rows otherwise, has no such reductions
@pytest.mark.parametrize("m_sizes,N,K,blocksize,rows,columns", [(TALL, 1184, 192, 64, 320, 192), (WIDE_MID, 1024, 64, 32, 256, 256),
                                                                (SQUARE, 1312, 192, 16, 256, 256),
                                                                (PAIR, 608, 192, 64, 160, 128)])
def test_packed_products(m_sizes, N, K, blocksize, rows, columns):
    c = Packed(m_sizes, N, K, blocksize)
    tile = ("pipe", rows, columns)
    y = check_tiles(lambda: grouped_gemm_forward_4bit(c.x, *c.w_q, c.ms), (*tile, FWD, True, 0))
    check_close(y, c.xw, what="forward")
    y = check_tiles(lambda: grouped_gemm_forward_4bit(c.x, *c.w_q, c.ms, torch.float32), (*tile, FWD, True, 0))
    check_close(y, c.xw, 1e-4, 1e-4, "forward, float32 result")
    src, idx, div = c.gather()
    y = check_tiles(lambda: grouped_gemm_forward_4bit_gathered(src, idx, div, *c.w_q, c.ms), (*tile, FWD, True, 0))
    assert torch.equal(y, grouped_gemm_forward_4bit(src[(idx // div).long()].contiguous(), *c.w_q, c.ms)), "gathered rows"
    y = check_tiles(lambda: grouped_gemm_forward_4bit_lora(c.x, *c.w_q, c.u, c.b, c.ms), (*tile, FWD, True, 2))
    check_close(y, c.xw + c.ub, what="forward, thin term")
    y = check_tiles(lambda: grouped_gemm_forward_4bit_lora(c.x, *c.w_q, c.u, c.b, c.ms, torch.float32), (*tile, FWD, True, 2))
    check_close(y, c.xw + c.ub, 1e-4, 1e-4, "forward, thin term, float32 result")
    dx = check_tiles(lambda: grouped_gemm_forward_transposed_4bit(c.x, *c.wt_q, c.ms), (*tile, DX, True, 0))
    check_close(dx, c.dx, what="input gradient")
    dx = check_tiles(lambda: grouped_gemm_forward_transposed_4bit(c.x, *c.wt_q, c.ms, torch.float32), (*tile, DX, True, 0))
    check_close(dx, c.dx, 1e-4, 1e-4, "input gradient, float32 result")
    dx = check_tiles(lambda: grouped_gemm_forward_transposed_4bit_lora(c.x, *c.wt_q, c.u, c.bt, c.ms), (*tile, DX, True, 2))
    check_close(dx, c.dx + c.ub, what="input gradient, thin term")
    dx = check_tiles(lambda: grouped_gemm_forward_transposed_4bit_lora(c.x, *c.wt_q, c.u, c.bt, c.ms, torch.float32),
                     (*tile, DX, True, 2))
    check_close(dx, c.dx + c.ub, 1e-4, 1e-4, "input gradient, thin term, float32 result")
    out = c.x2w2.astype(np.float32)
    out_dev = torch.from_numpy(out).to(DEV).bfloat16()
    start = to_np32(out_dev).astype(np.float64)
    check_tiles(lambda: grouped_gemm_forward_transposed_4bit(c.x, *c.wt_q, c.ms, out=out_dev, accumulate=True),
                (*tile, DX, True, 0))
    check_close(out_dev, start + c.dx, what="input gradient, accumulated")


@pytest.mark.parametrize("m_sizes,N,K,blocksize,rows,columns", [(TALL, 608, 192, 64, 320, 192), (SQUARE, 1312, 64, 32, 256, 256),
                                                                (PAIR, 296, 192, 64, 160, 128)])
def test_packed_gated_products(m_sizes, N, K, blocksize, rows, columns):
    c = Packed(m_sizes, N, K, blocksize)
    tile = ("pipe", rows, columns, FWD, True, 1)
    h, e, g = check_tiles(lambda: grouped_glu_forward_4bit(c.x, *c.w_q, *c.w2_q, c.ms, return_products=True), tile)
    check_close(e, c.xw, what="gate")
    check_close(g, c.xw2, what="up")
    assert torch.equal(h, silu_mul_forward(e, g))
    src, idx, div = c.gather()
    h = check_tiles(lambda: grouped_glu_forward_4bit(src, *c.w_q, *c.w2_q, c.ms, idx, div), tile)
    x = src[(idx // div).long()].contiguous()
    assert torch.equal(h, silu_mul_forward(grouped_gemm_forward_4bit(x, *c.w_q, c.ms),
                                           grouped_gemm_forward_4bit(x, *c.w2_q, c.ms)))
