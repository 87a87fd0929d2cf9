"""The sparse block as one library call each way against the block module by module: the same kernels, so the same bits
forward; backward the input gradient's two terms are summed before rounding instead of after."""
from types import SimpleNamespace

import pytest
import torch

from util import gen

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.modular_qwen3_moe_fused import MoeFusedLinear, Qwen3MoeFusedSparseMoeBlock  # noqa: E402
from qwen3_moe_fused.quantize.layer import MoeFusedLinear4bit  # noqa: E402

PROJ = ("gate_proj", "up_proj", "down_proj")


def _block(e, k, h, i, kind, seed):
    cfg = SimpleNamespace(num_experts=e, num_experts_per_tok=k, norm_topk_prob=seed % 2 == 0, hidden_size=h,
                          moe_intermediate_size=i, hidden_act="silu")
    dtype = torch.float32 if kind == "fp32" else torch.bfloat16
    blk = Qwen3MoeFusedSparseMoeBlock(cfg)
    with torch.no_grad():
        for p in blk.parameters():
            p.copy_(torch.randn(p.shape, generator=gen(seed + p.numel() % 89)) * p.shape[-1] ** -0.5)
    blk = blk.to(device="cuda", dtype=dtype)
    if kind.startswith("nf4"):
        for name in PROJ:
            old = getattr(blk, name)
            setattr(blk, name, MoeFusedLinear4bit(old.in_features, old.out_features, e, weight=old.weight, quant_type="nf4",
                                                  compress_statistics=kind == "nf4dq").cuda())
    return blk, dtype


SHAPES = [(1, 8, 2, 64, 32), (7 * 13, 11, 3, 16, 3), (65, 16, 1, 128, 64), (300, 8, 8, 256, 96), (129, 600, 4, 64, 64)]


@pytest.mark.parametrize("t,e,k,h,i", SHAPES)
@pytest.mark.parametrize("kind", ["bf16", "fp32"])
def test_block_call_both_ways(t, e, k, h, i, kind):
    blk, dtype = _block(e, k, h, i, kind, t)
    blk.keep_routing = True
    hidden = torch.randn((1, t, h), generator=gen(t)).to(dtype).cuda()
    dout = torch.randn((1, t, h), generator=gen(t + 1)).to(dtype).cuda()
    got = []
    for fused in (True, False):
        blk.fuse_front = fused
        with torch.no_grad():
            inferred = blk(hidden)[0]
        for frozen in ((), PROJ, ("gate", "up_proj")):
            for name in PROJ + ("gate",):
                getattr(blk, name).weight.requires_grad_(name not in frozen)
            blk.zero_grad(set_to_none=True)
            x = hidden.clone().requires_grad_(frozen != ("gate", "up_proj"))
            out, logits = blk(x)
            assert torch.equal(out, inferred)
            out.backward(dout)
            assert (x.grad is None) != x.requires_grad
            got.append([out, logits, blk.last_selected, x.grad] + [getattr(blk, n).weight.grad for n in PROJ + ("gate",)])
    tol = 1e-5 if kind == "fp32" else 2e-2
    for a, b in zip(got[:3], got[3:]):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])
        for u, v in zip(a[3:], b[3:]):
            assert (u is None) == (v is None)
            if u is not None:
                scale = float(v.abs().max()) or 1.0
                assert float((u.float() - v.float()).abs().max()) <= tol * scale


# (two times t tokens; the first five: the down projection and the sum over the selections in one launch, up to 16 selections)
@pytest.mark.parametrize("t,e,k,h,i", [(1, 8, 2, 256, 512), (1, 16, 8, 128, 768), (1, 32, 8, 192, 576), (4, 24, 2, 128, 768),
                                       (1, 16, 5, 64, 320), (3, 8, 2, 128, 384), (9, 16, 4, 512, 128), (200, 8, 4, 128, 96), (1500, 6, 2, 128, 256)])
@pytest.mark.parametrize("kind", ["nf4", "nf4dq"])
def test_block_call_on_packed_weights(t, e, k, h, i, kind):
    blk, dtype = _block(e, k, h, i, kind, t)
    hidden = torch.randn((2, t, h), generator=gen(t)).to(dtype).cuda()
    out = []
    for fused in (True, False):
        blk.fuse_front = fused
        with torch.no_grad():
            out.append(blk(hidden)[0].float())
    # up to 128 rows per expert both run on the same kernels; beyond, the gated product and the two plain ones round in
    # another place (a bf16 step of the product, 2^-8 of its size, through the unit and the down projection)
    if 2 * t * k <= 128 * e:
        assert torch.equal(out[0], out[1])
    assert float((out[0] - out[1]).abs().max()) <= 2e-2 * float(out[1].abs().max())


# blocks of 32: an inner size that is no multiple of 64 has another down projection, and its sum over the selections by itself
@pytest.mark.parametrize("i", [288, 480, 320, 512])
@pytest.mark.parametrize("kind", ["nf4", "nf4dq"])
def test_block_call_on_packed_weights_in_blocks_of_32(i, kind):
    from qwen3_moe_fused.quantize.layer import Nf4Params
    from qwen3_moe_fused.quantize.nf4 import quantize_nf4

    blk, dtype = _block(8, 2, 128, i, kind, 1)
    for seed, name in enumerate(PROJ):
        proj = getattr(blk, name)
        w = torch.randn((8, proj.out_features, proj.in_features), generator=gen(seed)) * proj.in_features ** -0.5
        packed, state = quantize_nf4(w.to(dtype).cuda(), 32, compress_statistics=kind == "nf4dq")
        proj._parameters["weight"] = Nf4Params(packed, quant_state=state)
    hidden = torch.randn((2, 1, 128), generator=gen(i)).to(dtype).cuda()
    out = []
    for fused in (True, False):
        blk.fuse_front = fused
        with torch.no_grad():
            out.append(blk(hidden)[0])
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])


def test_block_call_on_two_streams_and_with_a_hook():
    blk, _ = _block(8, 2, 64, 64, "bf16", 3)
    xs = [torch.randn((1, 40, 64), generator=gen(s)).to(torch.bfloat16).cuda() for s in range(2)]
    with torch.no_grad():
        want = [blk(x)[0] for x in xs]
        streams = [torch.cuda.Stream() for _ in xs]
        torch.cuda.synchronize()
        got = []
        for x, s in zip(xs, streams):
            with torch.cuda.stream(s):
                got.append([blk(x)[0] for _ in range(5)])
        torch.cuda.synchronize()
        assert all(torch.equal(g, w) for gs, w in zip(got, want) for g in gs)
        seen = []
        handle = blk.down_proj.register_forward_hook(lambda m, a, o: seen.append(o.shape))
        assert torch.equal(blk(xs[0])[0], want[0]) and len(seen) == 1
        handle.remove()
    assert type(blk.down_proj) is MoeFusedLinear


def test_block_call_leaves_hooks_forward_mode_and_the_routing_alone():
    blk, _ = _block(8, 2, 64, 64, "fp32", 5)
    blk.keep_routing = True
    x = torch.randn((1, 40, 64), generator=gen(5)).cuda()
    with torch.no_grad():
        want = blk(x)[0]
        assert blk.last_selected.untyped_storage().nbytes() == 40 * 2 * 8
        seen = []
        handle = blk.up_proj.register_forward_hook(lambda m, a, o: seen.append(o.shape))
        assert torch.equal(blk(x)[0], want) and len(seen) == 1
        handle.remove()
        with torch.autograd.forward_ad.dual_level(), pytest.raises(Exception):  # no kernel here has a forward-mode rule
            blk(torch.autograd.forward_ad.make_dual(x, x))


@pytest.mark.parametrize("kind", ["bf16", "nf4dq"])
def test_rows_beyond_one_call(kind, monkeypatch):
    """The same bits on both sides of the row count that ends the one call."""
    blk, dtype = _block(8, 4, 256, 128, kind, 4)
    hidden = torch.randn((1, 33, 256), generator=gen(4)).to(dtype).cuda()
    got = []
    for rows in (33 * 4, 33 * 4 - 1):
        monkeypatch.setattr(blk, "_ONE_CALL_ROWS", rows, raising=False)
        with torch.no_grad():
            assert (blk._one_call(hidden[0], blk.gate(hidden[0])) is None) == (rows < 33 * 4)
            got.append(blk(hidden))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def _apart(t):
    """The same values with the last dimension's elements two apart."""
    return torch.stack((t, torch.zeros_like(t)), dim=-1)[..., 0]


def _shifted(t):
    """The same values one element past where an allocation starts."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


@pytest.mark.parametrize("unpack", [_apart, _shifted])
@pytest.mark.parametrize("kind", ["bf16", "fp32"])
def test_block_call_with_saved_tensors_handed_back_elsewhere(unpack, kind):
    """Saved-tensor hooks (offloading, packing into one buffer) hand back equal tensors, not the same ones."""
    blk, dtype = _block(8, 2, 64, 64, kind, 6)
    grads = []
    for hooks in ((lambda t: t, lambda t: t), (lambda t: t.clone(), unpack)):
        x = torch.randn((1, 700, 64), generator=gen(6)).to(dtype).cuda().requires_grad_()
        blk.zero_grad(set_to_none=True)
        with torch.autograd.graph.saved_tensors_hooks(*hooks):
            out, logits = blk(x)
        (out.float().square().sum() + logits.float().sum()).backward()
        grads.append([x.grad] + [p.grad for p in blk.parameters()])
    for a, b in zip(*grads):
        assert float((a.float() - b.float()).abs().max()) <= (1e-5 if kind == "fp32" else 2e-2) * float(a.float().abs().max())


# one side as thin as an adapter's rank, the other a multiple of 256, 16384 rows and more: the rows are dealt out evenly
@pytest.mark.parametrize("t,k,h,i", [(8192, 2, 256, 32), (5500, 3, 512, 64), (16500, 1, 16, 256)])
def test_block_call_deals_the_rows_of_thin_weight_gradients_out(t, k, h, i):
    """The same bits as the separate steps, whose weight gradients take the kernel with even shares."""
    blk, dtype = _block(8, k, h, i, "bf16", 2)
    with torch.no_grad():
        blk.gate.weight[0] += 0.1  # one popular expert
    x, dout = (torch.randn((1, t, h), generator=gen(s)).abs().to(dtype).cuda() for s in (1, 2))
    grads = []
    for fused in (True, False):
        blk.zero_grad(set_to_none=True)
        blk._ONE_CALL_ROWS = 65536 if fused else 0
        blk(x)[0].backward(dout)
        grads.append([getattr(blk, n).weight.grad for n in PROJ])
    assert all(torch.equal(a, b) for a, b in zip(*grads))
