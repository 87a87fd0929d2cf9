"""Joining and splitting two adapters' thin matrices against torch's own concatenation, bit for bit."""
import ctypes

import pytest
import torch

from util import gen

pytestmark = pytest.mark.gpu

from qwen3_moe_fused import _lib  # noqa: E402
from qwen3_moe_fused.kernels.fast_lora import _copy_pieces, _halves, _joined, _padded  # noqa: E402


# runs of one piece of 16 bytes and less (the stock copies), of odd counts, of unequal ranks, around the 1024 pieces of a
# workgroup; no experts at all
@pytest.mark.parametrize("e,ra,rb,h", [(3, 8, 8, 8), (5, 4, 4, 40), (7, 16, 8, 264), (1, 1, 3, 5), (2, 16, 16, 4096), (128, 32, 32, 96),
                                       (0, 8, 8, 16), (33, 24, 8, 31)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_join_pad_and_split(e, ra, rb, h, dtype):
    g = gen(e + h)
    a, b = (torch.randn((e, r, h), generator=g).to(dtype).cuda() for r in (ra, rb))
    u, v = (torch.randn((e * 3, r), generator=g).to(dtype).cuda() for r in (ra, rb))
    p, q = (torch.randn((e, h, r), generator=g).to(dtype).cuda() for r in (ra, rb))
    pieces = []
    got = [_joined(a, b, 1, pieces), _joined(u, v, 1, pieces), _padded(p, 2, 0, ra + rb, pieces), _padded(q, 2, ra, ra + rb, pieces)]
    _copy_pieces(pieces, True)
    want = [torch.cat((a, b), 1), torch.cat((u, v), 1), torch.cat((p, torch.zeros_like(q)), 2), torch.cat((torch.zeros_like(p), q), 2)]
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    for wide, parts in ((got[0], (a, b)), (got[1], (u, v))):
        halves = _halves(wide, 1, ra)
        assert all(torch.equal(x, y) and x.is_contiguous() for x, y in zip(halves, parts))


def test_strided_and_mixed_operands():
    g = gen(3)
    a, b = (torch.randn((5, 24, 16), generator=g).bfloat16().cuda().transpose(1, 2) for _ in range(2))
    p = torch.randn((5, 16, 24), generator=g).bfloat16().cuda().transpose(1, 2)
    f = torch.randn((5, 16, 24), generator=g).cuda()
    pieces = []
    got = [_joined(a, b, 1, pieces), _padded(p, 2, 0, 32, pieces), _joined(a, f, 1, pieces)]
    _copy_pieces(pieces, True)
    want = [torch.cat((a, b), 1), torch.cat((p, torch.zeros_like(p)), 2), torch.cat((a, f), 1)]
    assert all(torch.equal(x, y) and x.dtype == y.dtype for x, y in zip(got, want))


def test_copy_blocks_refuses_what_it_cannot_copy():
    buf = torch.zeros(256, device="cuda", dtype=torch.uint8)
    at = buf.data_ptr()

    def call(*jobs):
        return _lib.lib().mfl_copy_blocks((_lib.BlockCopy * len(jobs))(*(_lib.BlockCopy(*j) for j in jobs)), len(jobs), _lib.stream())

    ok = (at, at + 128, 2, 16, 16, 16)
    assert call(ok) == 0 and call((None, at, 0, 16, 16, 16)) == 0 and call(*[ok] * 8) == 0
    assert call(*[ok] * 9) == -6 and call((at, at + 128, 2, 8, 16, 16)) == -6 and call((at + 4, at + 128, 1, 16, 16, 16)) == -6
    assert call((at, at + 128, 1 << 20, 1 << 20, 16, 16)) == -6
    assert call((at, None, 1, 16, 16, 16)) != 0 and call((at, at + 128, -1, 16, 16, 16)) != 0
    assert _lib.lib().mfl_copy_blocks(ctypes.POINTER(_lib.BlockCopy)(), 1, _lib.stream()) != 0
