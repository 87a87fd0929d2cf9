"""The shape- and type-generic kernel (fp32 / fp16 operands, dimensions that are no multiple of 8) at the edges of its
tiles, against float64 sums.

Tolerance: an fp32 sum of L products in any order is within L * 2^-24 * sum |a b| of the exact one (each of the L - 1
additions and L products rounds once); ``alpha``, the old value of an accumulated output and the final rounding add one
unit in the last place of the output type each."""
import pytest
import torch

from util import gen

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.grouped_gemm.backward_dw import grouped_gemm_backward_dw  # noqa: E402
from qwen3_moe_fused.grouped_gemm.forward import grouped_gemm_forward  # noqa: E402
from qwen3_moe_fused.grouped_gemm.forward_transposed import grouped_gemm_forward_transposed  # noqa: E402

ULP = {torch.float32: 2.0 ** -23, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


def _check(got, exact, bound, length, alpha, old, what):
    ulp = ULP[got.dtype]
    exact = alpha * exact + (0 if old is None else old.double())
    room = length * 2.0 ** -24 * abs(alpha) * bound + 2 * ulp * (exact.abs() + (0 if old is None else old.double().abs()))
    diff = (got.double().cpu() - exact).abs()
    assert torch.isfinite(got).all()
    assert (diff <= room + 1e-30).all(), f"{what}: {float((diff - room).max()):.3e} over the bound"


def _products(x, w, dy, sizes):
    """(y, dx, dw) and the same of the operands' absolute values, float64 on the CPU."""
    x, w, dy = x.double(), w.double(), dy.double()
    y, dx, dw, o = [], [], [], 0
    for e, m in enumerate(sizes):
        xe, de = x[o:o + m], dy[o:o + m]
        y.append(xe @ w[e].t()), dx.append(de @ w[e]), dw.append(de.t() @ xe)
        o += m
    return torch.cat(y), torch.cat(dx), torch.stack(dw)


# row counts on both sides of the 16-, 32- and 64-row tiles; N and K on both sides of the tiles' columns, of a reduction
# step (16, 64, 128) and of the groups of four that are loaded at once
CASES = [
    ([1, 0, 16, 17, 5], 32, 128),          # 16-row tiles, whole ones
    ([15, 33, 0, 2], 33, 132),             # ... a ragged last column tile, one reduction group past a step
    ([16, 16, 1], 70, 257),                # ... sizes that are no multiple of four
    ([31, 33, 64, 0, 1], 64, 64),          # 32-row tiles
    ([40, 65, 2], 129, 131),
    ([700, 300], 4160, 24),                # 64-row tiles (enough of them to fill the chip twice over)
    ([513, 500], 4097, 23),
    ([3, 0, 200, 1], 16, 68),              # weight gradient with a side of 16
    ([9, 40], 15, 7),
    ([17, 0, 15, 33], 65, 129),            # weight gradient: 64 x 128 tiles, steps of 16 rows
    ([64], 3, 1),
]


@pytest.mark.parametrize("sizes,n,k", CASES)
@pytest.mark.parametrize("dtype,out", [(torch.float32, torch.float32), (torch.float16, torch.float32),
                                       (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("alpha,accumulate", [(1.0, False), (0.5, True)])
def test_generic_products_within_the_bound_of_their_sums(sizes, n, k, dtype, out, alpha, accumulate):
    g = gen(sum(sizes) + n + k)
    rows, experts = sum(sizes), len(sizes)
    mk = lambda *s: torch.randn(s, generator=g).to(dtype)
    x, w, dy = mk(rows, k), mk(experts, n, k), mk(rows, n)
    ms = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    exact = _products(x, w, dy, sizes)
    bound = _products(x.abs(), w.abs(), dy.abs(), sizes)
    xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
    longest = max(sizes)
    for i, (fn, args, length) in enumerate(((grouped_gemm_forward, (xd, wd, ms), k),
                                            (grouped_gemm_forward_transposed, (dyd, wd, ms), n),
                                            (grouped_gemm_backward_dw, (xd, dyd, ms), longest))):
        old = torch.randn(exact[i].shape, generator=g).to(out) if accumulate else None
        # one element past a 16-byte boundary: the stores fall back to single elements
        res = torch.full((exact[i].numel() + 1,), float("nan"), dtype=out, device="cuda")[1 if n % 2 else 0:]
        res = res[:exact[i].numel()].view(exact[i].shape)
        if accumulate:
            res.copy_(old)
        got = fn(*args, out, out=res, alpha=alpha, accumulate=accumulate)
        _check(got, exact[i], bound[i], length, alpha, old, fn.__name__)


# short reductions (a step of 16, up to it, past it; aligned outputs and odd ones), up to 128 with tiles enough to fill the
# chip, fp16 in odd sizes, weight gradients of a few rows (n x k as outputs: on both sides of the tiles' columns)
SHORT = [
    ([5, 0, 30], 132, 16),
    ([5, 0, 30], 129, 15),
    ([70, 60], 200, 17),
    ([70, 60], 201, 32),
    ([700, 300], 4160, 4),
    ([700, 300], 4161, 16),
    ([700, 300], 4161, 31),
    ([700, 300], 4164, 33),
    ([700, 320], 4161, 128),
    ([3000, 1100], 2049, 131),
    ([1], 130, 260),
    ([3, 0, 1, 2], 65, 129),
    ([16, 0], 128, 128),
]


@pytest.mark.parametrize("sizes,n,k", SHORT)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_short_reductions_and_few_rows_within_the_bound(sizes, n, k, dtype):
    for length in ((n, k), (k, n)):  # the forward's short reduction, then the input gradient's
        test_generic_products_within_the_bound_of_their_sums(sizes, *length, dtype, torch.float32, 0.5, True)


@pytest.mark.parametrize("n", [65535 * 32, 65535 * 32 + 1, 65535 * 64])
def test_outputs_of_more_column_tiles_than_a_grid_has_rows(n):
    """The narrowest tiles are left to the wider ones where their number would pass 65535: one row, short and longer sums."""
    ms = torch.tensor([1], dtype=torch.int32, device="cuda")
    torch.manual_seed(n)
    for k, fn in ((4, grouped_gemm_forward), (3, grouped_gemm_forward_transposed), (36, grouped_gemm_forward),
                  (35, grouped_gemm_forward_transposed)):
        a = torch.randn((1, k), device="cuda")
        w = torch.randn((1, n, k) if fn is grouped_gemm_forward else (1, k, n), device="cuda")
        got = fn(a, w, ms, torch.float32)[0].double()
        exact, bound = torch.zeros_like(got), torch.zeros_like(got)
        for j in range(k):
            term = a[0, j].double() * (w[0, :, j] if fn is grouped_gemm_forward else w[0, j]).double()
            exact += term
            bound += term.abs()
        assert ((got - exact).abs() <= k * 2.0 ** -24 * bound + 2.0 ** -23 * exact.abs()).all()


# Matrices larger than the last cache, rows of whole lines: the weights are loaded, a weight gradient is stored past the
# caches.  Tiles of 16 and of 32 rows, experts without rows, one with a second tile, output tiles that end inside both ways.
@pytest.mark.parametrize("sizes", [[8, 0, 17, 1] * 8 + [16], [20, 33, 0, 24] * 8 + [31]])
def test_matrices_larger_than_the_caches(sizes):
    e, n, k, rows = len(sizes), 1056, 2080, sum(sizes)
    assert e * n * k * 4 > 256 << 20
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, dy = (torch.randn((rows, c), device="cuda", generator=g) for c in (k, n))
    w = torch.randn((e, n, k), device="cuda", generator=g)
    ms = torch.tensor(sizes, dtype=torch.int32).cuda()
    got = (grouped_gemm_forward(x, w, ms), grouped_gemm_forward_transposed(dy, w, ms), grouped_gemm_backward_dw(x, dy, ms, torch.float32))
    for y, exact, bound, length, what in zip(got, _products(x, w, dy, sizes), _products(x.abs(), w.abs(), dy.abs(), sizes),
                                             (k, n, max(sizes)), ("forward", "dx", "dw")):
        room = length * 2.0 ** -24 * bound + 2 * ULP[torch.float32] * exact.abs()
        assert torch.isfinite(y).all() and ((y.double() - exact).abs() <= room + 1e-30).all(), what
