"""Double-quantised NF4 weights, whose 8-bit scales the decode-sized kernels read as they are: the same bits as with the
scales written out in fp32 first (code256[q] * absmax2 rounded, then the offset added and rounded, in both)."""
import pytest
import torch

from util import gen

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.grouped_gemm.forward_4bit import grouped_gemm_forward_4bit  # noqa: E402
from qwen3_moe_fused.grouped_gemm.fused import grouped_gemm_forward_4bit_gathered, grouped_glu_forward_4bit  # noqa: E402
from qwen3_moe_fused.quantize.nf4 import Nf4QuantState, _quantize_absmax, quantize_nf4, resolve_absmax  # noqa: E402
from qwen3_moe_fused.quantize.nf4 import write_out_scales  # noqa: E402


def _weights(e, n, k, blocksize, seed):
    w = (torch.randn((e, n, k), generator=gen(seed)) * 0.02).to(torch.bfloat16).cuda()
    packed, nested = quantize_nf4(w, blocksize, "nf4", compress_statistics=True)
    assert nested.nested
    plain = Nf4QuantState(absmax=resolve_absmax(nested), shape=nested.shape, code=nested.code, blocksize=blocksize)
    return packed, nested, plain


@pytest.mark.parametrize("n", [1, 15, 16, 255, 256, 257, 4096, 100003])
@pytest.mark.parametrize("blocksize2", [8, 256])
def test_scales_written_out_are_the_formula(n, blocksize2):
    from qwen3_moe_fused.quantize.nf4 import BlockwiseState

    g = gen(n)
    q = torch.randint(0, 256, (n,), generator=g, dtype=torch.uint8).cuda()
    code = torch.randn(256, generator=g).cuda()
    absmax2 = torch.rand((n + blocksize2 - 1) // blocksize2, generator=g).cuda()
    offset = torch.tensor(0.0473).cuda()
    state = Nf4QuantState(absmax=q, shape=(1,), code=code, offset=offset,
                          state2=BlockwiseState(absmax=absmax2, code=code, blocksize=blocksize2))
    want = code[q.long()] * absmax2.repeat_interleave(blocksize2)[:n] + offset
    assert torch.equal(resolve_absmax(state), want)


# (rows per expert, N, K, blocksize): the matrix-vector kernel (up to two rows per expert; rows of at most 1024, and of
# more), the streaming kernel with 32-row and 64-row tiles; rows of the matrix that cross a border of the second-level
# blocks (K = 768: 12 scales a row), column tiles that end past N, scales under blocks of 128, a row of more scales than a
# second-level block (no kernel for it), and batches beyond the decode sizes
CASES = [
    ([1, 0, 1, 2, 0, 0, 0, 0, 0], 64, 2048, 64),
    ([1, 0, 1, 0, 0], 96, 768, 64),
    ([2, 1, 0, 2], 32, 1536, 64),
    ([1, 1, 0], 32, 1024, 128),
    ([1, 0, 2, 1], 64, 768, 64),
    ([1, 0, 1], 128, 576, 64),
    ([2, 0, 1, 0], 64, 320, 64),
    ([1, 2, 0, 3], 64, 960, 64),
    # blocks smaller than a lane's run
    ([1, 0, 2, 1], 64, 2048, 8),
    ([1, 0, 2, 1], 64, 1024, 16),
    ([1, 2, 0, 1], 64, 768, 32),
    ([1, 0, 2, 1], 64, 512, 16),
    ([5, 0, 3, 17], 200, 768, 64),
    ([40, 1, 33], 128, 384, 64),
    ([70, 0, 12], 72, 2048, 64),
    ([9], 40, 16512, 64),
    ([4, 9], 64, 256, 128),
    ([600, 20], 64, 256, 64),
    # stages that do not divide by eight or two, and more of them than the registers hold at once, at both tile heights
    ([5, 30], 160, 2176, 64),
    ([5, 30], 72, 4224, 64),
    ([50, 3], 96, 4096, 64),
    ([40, 30], 40, 2432, 64),
]


@pytest.mark.parametrize("sizes,n,k,blocksize", CASES)
def test_products_on_double_quantised_weights_are_those_on_written_out_scales(sizes, n, k, blocksize):
    e, rows = len(sizes), sum(sizes)
    gate, gate_nested, gate_plain = _weights(e, n, k, blocksize, n + k)
    up, up_nested, up_plain = _weights(e, n, k, blocksize, n + k + 1)
    ms = torch.tensor(sizes, dtype=torch.int32).cuda()
    src = torch.randn((rows, k), generator=gen(rows)).to(torch.bfloat16).cuda()
    idx = torch.randperm(rows, generator=gen(rows + 1)).to(torch.int32).cuda()
    for dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(grouped_gemm_forward_4bit(src, gate, gate_nested, ms, dtype),
                           grouped_gemm_forward_4bit(src, gate, gate_plain, ms, dtype))
    assert torch.equal(grouped_gemm_forward_4bit_gathered(src, idx, 1, gate, gate_nested, ms),
                       grouped_gemm_forward_4bit_gathered(src, idx, 1, gate, gate_plain, ms))
    got = grouped_glu_forward_4bit(src, gate, gate_nested, up, up_nested, ms, idx, 1, return_products=True)
    want = grouped_glu_forward_4bit(src, gate, gate_plain, up, up_plain, ms, idx, 1, return_products=True)
    for a, b in zip(got, want):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("blocksize2", [1, 3, 100])
def test_second_level_blocks_of_any_size(blocksize2):
    from qwen3_moe_fused.fused_mlp import moe_block_4bit
    from qwen3_moe_fused.quantize.layer import Nf4Params
    from qwen3_moe_fused.quantize.nf4 import _quantize_absmax

    e, k, n, rows = 3, 128, 64, 10
    states = []
    for seed, shape in enumerate(((e, n, k), (e, n, k), (e, k, n))):
        packed, state = quantize_nf4((torch.randn(shape, generator=gen(seed)) * 0.02).to(torch.bfloat16).cuda(), 64)
        q, state2, offset = _quantize_absmax(state.absmax, blocksize2)
        nested = Nf4QuantState(absmax=q, shape=shape, code=state.code, blocksize=64, offset=offset, state2=state2)
        want = state2.code[q.long()] * state2.absmax.repeat_interleave(blocksize2)[:q.numel()] + offset
        plain = Nf4QuantState(absmax=want, shape=shape, code=state.code, blocksize=64)
        assert torch.equal(resolve_absmax(nested), want)
        states.append((packed, nested, plain))
    x = torch.randn((rows, k), generator=gen(9)).to(torch.bfloat16).cuda()
    ms = torch.tensor([4, 0, 6], dtype=torch.int32).cuda()
    idx = torch.randperm(rows, generator=gen(8)).to(torch.int32).cuda()
    (g, g8, g32), (u, u8, u32), (d, d8, d32) = states
    assert torch.equal(grouped_gemm_forward_4bit(x, g, g8, ms), grouped_gemm_forward_4bit(x, g, g32, ms))
    assert torch.equal(grouped_gemm_forward_4bit_gathered(x, idx, 1, g, g8, ms),
                       grouped_gemm_forward_4bit_gathered(x, idx, 1, g, g32, ms))
    assert torch.equal(grouped_glu_forward_4bit(x, g, g8, u, u8, ms, idx, 1), grouped_glu_forward_4bit(x, g, g32, u, u32, ms, idx, 1))
    logits = torch.randn((rows, e), generator=gen(7)).to(torch.bfloat16).cuda()
    outs = [moe_block_4bit(x, logits, *(Nf4Params(p, quant_state=s) for p, s in zip((g, u, d), which)), 2, True)[0]
            for which in ((g8, u8, d8), (g32, u32, d32))]
    assert torch.equal(*outs)


# several matrices' scales in one launch: sizes that differ, one that four does not divide, a plain state and none between them
def test_scales_of_several_matrices_written_out_at_once():
    states = []
    for n, blocksize2 in ((3 * 8 * 64, 256), (1 * 7 * 64, 8), (2 * 96 * 192, 256)):
        _, nested, _ = _weights(1, n // 64, 64, 64, n)
        if blocksize2 != 256:
            scales = resolve_absmax(nested)
            nested.absmax, nested.state2, nested.offset = _quantize_absmax(scales, blocksize2)
        states.append(nested)
    plain = _weights(1, 8, 64, 64, 5)[2]
    got = write_out_scales(states[0].absmax, states[0], plain, None, states[1], states[2])
    assert got[1] is plain and got[2] is None
    for state, out in zip(states, (got[0], got[3], got[4])):
        assert not out.nested and torch.equal(out.absmax, resolve_absmax(state))
