"""The tiles of the row-grouped bf16 products: which of them a product runs on, from the names of the launched kernels."""
import numpy as np
import pytest
import torch

import oracle
from util import check_close, check_tiles, gen, randn, to_np32

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.grouped_gemm.fused import grouped_glu_forward  # noqa: E402
from qwen3_moe_fused.kernels.silu_mul import silu_mul_forward  # noqa: E402

DEV = "cuda"
FWD = 0


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
