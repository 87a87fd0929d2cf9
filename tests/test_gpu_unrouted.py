"""Tokens whose logits are NaN select no expert: the sort places their selections behind all others, and the block's
results for the other tokens, and the memory around its tensors, are what they are without such tokens."""
import numpy as np
import pytest
import torch

from util import gen, randn

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.kernels.indexing import get_expert_counts_and_idx  # noqa: E402
from qwen3_moe_fused.kernels.routing import route_and_sort  # noqa: E402
from test_gpu_block_call import PROJ, _block  # noqa: E402

DEV = "cuda"


def _check_sort(keys, E, counts, sort_idx, inv):
    keys = np.where((keys < 0) | (keys >= E), E, keys)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(counts.cpu().numpy(), np.bincount(keys, minlength=E + 1)[:E])
    assert np.array_equal(sort_idx.cpu().numpy(), order)
    assert np.array_equal(inv.cpu().numpy(), np.argsort(order))


# one workgroup (up to 32 tokens), two launches, three launches (more than 512 experts)
@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (5, 128, 8), (32, 512, 64), (33, 128, 8), (1000, 60, 3), (4096, 128, 8),
                                   (300, 600, 4)])
@pytest.mark.parametrize("bad", [(0,), (-1,), (0.5, 0.51, -1), "all"])
def test_selections_of_nan_rows_come_last(T, E, k, bad):
    logits = randn((T, E), gen(T + E), 2.0)
    rows = range(T) if bad == "all" else [min(T - 1, int(b * T)) if b >= 0 else T - 1 for b in bad]
    for r in rows:
        logits[r] = float("nan")
    for renorm in (True, False):
        w, sel, m_sizes, sort_idx, inv = route_and_sort(logits.to(DEV), k, renorm, torch.bfloat16, E)
        sel = sel.cpu().numpy()
        assert all((sel[r] == 0x7FFFFFFF).all() for r in rows)
        _check_sort(sel.reshape(-1), E, m_sizes, sort_idx, inv)
        nan = np.zeros(T, bool)
        nan[list(rows)] = True
        assert np.array_equal(torch.isnan(w).all(1).cpu().numpy(), nan) and not torch.isnan(w[~nan]).any()


# the two-kernel sort (up to 512 experts), one workgroup, several workgroups
@pytest.mark.parametrize("R,E", [(1, 4), (63, 128), (5000, 128), (300000, 7), (3000, 600), (70000, 600)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_ids_outside_the_range_come_last(R, E, dtype):
    sel = torch.randint(-1, E + 1, (R,), generator=gen(R + E)).to(dtype)
    counts, sort_idx, inv = get_expert_counts_and_idx(sel.to(DEV), E)
    _check_sort(sel.numpy(), E, counts, sort_idx, inv)


def _close(a, b, tol):
    assert float((a.float() - b.float()).abs().max()) <= tol * max(1e-3, float(b.float().abs().max()))


# one row per expert and more, one selection per token and more; the packed weights' three kernels, and (the third and fourth) the
# down projection with the sum over the selections in one launch
@pytest.mark.parametrize("t,e,k,h,i", [(1, 8, 2, 64, 32), (3, 16, 4, 512, 128), (1, 8, 2, 64, 512), (3, 16, 5, 512, 768), (65, 16, 1, 128, 64), (300, 8, 8, 256, 96)])
@pytest.mark.parametrize("kind", ["bf16", "fp32", "nf4", "nf4dq"])
@pytest.mark.parametrize("one_call", [True, False])
def test_block_with_a_nan_token(t, e, k, h, i, kind, one_call):
    blk, dtype = _block(e, k, h, i, kind, 2 * t)
    blk.fuse_front = one_call
    bad = t // 2
    keep = torch.arange(t, device=DEV) != bad
    clean = torch.randn((1, t, h), generator=gen(t)).to(dtype).to(DEV)
    broken = clean.clone()
    broken[0, bad, 1] = float("nan")
    with torch.no_grad():
        want, got = blk(clean)[0][0], blk(broken)[0][0]
    tol = 1e-5 if kind == "fp32" else 2e-2
    assert torch.isnan(got[bad]).all()
    if t > 1:
        _close(got[keep], want[keep], tol)
    if kind.startswith("nf4"):
        return
    dout = torch.randn((1, t, h), generator=gen(t + 1)).to(dtype).to(DEV)
    quiet = dout.clone()
    quiet[0, bad] = 0  # what the token adds to the experts' gradients without its NaN
    grads = []
    for x, d in ((clean, quiet), (broken, dout)):
        x = x.clone().requires_grad_()
        blk.zero_grad(set_to_none=True)
        blk(x)[0].backward(d)
        grads.append([x.grad[0][keep]] + [getattr(blk, n).weight.grad for n in PROJ])
        assert torch.isnan(x.grad[0][bad]).all() == (x.isnan().any())
    for want, got in zip(*grads):
        if want.numel():
            _close(got, want, tol)
