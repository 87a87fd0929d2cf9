"""The forms of the routing and combine kernels that few tokens take, at the edges of their ranges."""
import numpy as np
import pytest
import torch

import oracle
from util import gen, randn

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.kernels.routing import combine_rows, route_and_sort  # noqa: E402

DEV = "cuda"


# one workgroup up to 32 tokens: 4, 8 or 16 waves; one to eight batches of 64 selections per wave
@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (4, 128, 8), (5, 65, 3), (8, 512, 64), (9, 64, 64), (31, 128, 1), (32, 512, 64),
                                   (33, 512, 64)])
@pytest.mark.parametrize("nan_row", [False, True])
def test_one_workgroup_routing(T, E, k, nan_row):
    logits = randn((T, E), gen(T + E), 2.0)
    keep = np.ones(T, bool)
    if nan_row:
        logits[T // 2] = float("nan")
        keep[T // 2] = False
    w, sel, m_sizes, sort_idx, inv = route_and_sort(logits.to(DEV), k, True, torch.float32, E)
    torch.cuda.synchronize()
    w_ref, sel_ref = oracle.softmax_topk(logits.numpy()[keep], k, True)
    sel_ref = np.asarray(sel_ref).reshape(-1, k)
    assert np.array_equal(sel.cpu().numpy()[keep], sel_ref)
    np.testing.assert_allclose(w.cpu().numpy()[keep], np.asarray(w_ref).reshape(-1, k), rtol=1e-5)
    counts, s_ref, i_ref = oracle.expert_counts_and_idx(sel_ref.reshape(-1), E) if keep.any() else (np.zeros(E), [], [])
    assert np.array_equal(m_sizes.cpu().numpy(), counts)
    n = int(keep.sum()) * k
    orig = np.nonzero(np.repeat(keep, k))[0]
    assert np.array_equal(sort_idx.cpu().numpy()[:n], orig[np.asarray(s_ref, dtype=np.int64)])
    assert np.array_equal(inv.cpu().numpy()[orig], i_ref)


# a wave per slice of 1 KiB up to 512 tokens, a wave per row beyond; more rows per token than are in flight, rows that
# end inside a slice, rows of no 16-byte multiple
@pytest.mark.parametrize("T", [1, 5, 512, 513])
@pytest.mark.parametrize("k,H,dtype", [(8, 2048, torch.bfloat16), (9, 520, torch.bfloat16), (3, 37, torch.bfloat16),
                                       (1, 260, torch.float32)])
def test_combine_against_fp64(T, k, H, dtype):
    g = gen(T + k + H)
    y, w = randn((T * k, H), g, 1.0, dtype), randn((T, k), g, 1.0, dtype)
    pos = torch.randperm(T * k, generator=g).to(torch.int32)
    got = combine_rows(y.to(DEV), pos.to(DEV), w.to(DEV), torch.argsort(pos).to(torch.int32).to(DEV)).double().cpu()
    terms = y.double()[pos.long()].view(T, k, H) * w.double().unsqueeze(-1)
    # k fused multiply-adds in fp32, then one rounding to the type
    room = (k * 2.0 ** -23) * terms.abs().sum(1) + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * terms.sum(1).abs()
    assert ((got - terms.sum(1)).abs() <= room).all()
