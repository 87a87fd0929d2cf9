"""The router projection and its gradients against float64 products.  Tolerance: fp32 sums of L products in any order are
within L * 2^-24 * sum |a b| of the exact ones, plus one bf16 rounding (2^-8 of the value)."""
import pytest
import torch

from util import gen

pytestmark = pytest.mark.gpu

from qwen3_moe_fused.kernels.routing import router_linear  # noqa: E402
from qwen3_moe_fused.modular_qwen3_moe_fused import Qwen3MoeFusedRouter  # noqa: E402


def _near(got, a, b, length, ulp=2.0 ** -8):
    exact, bound = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    room = length * 2.0 ** -24 * bound + ulp * exact.abs()
    assert torch.isfinite(got).all() and ((got.double().cpu() - exact).abs() <= room + 1e-30).all()


# tokens around the blocks of 16 and 64 of the forward, the steps of 32 and parts of 256 of the weight gradient; experts
# around the blocks of 16 and 128; hidden sizes of one piece, of pieces that do not divide among eight waves, of a last
# column tile that is not whole
@pytest.mark.parametrize("t,h,e", [(1, 2048, 128), (15, 64, 8), (16, 576, 16), (17, 1024, 136), (33, 512, 60), (64, 192, 8),
                                   (255, 264, 128), (257, 2048, 120), (511, 640, 264), (512, 264, 128), (513, 2048, 120), (769, 136, 264), (3001, 128, 64)])
def test_router_projection_and_gradients(t, h, e):
    g = gen(t + h + e)
    x, w, d = (torch.randn(s, generator=g).to(torch.bfloat16) for s in ((t, h), (e, h), (t, e)))
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    y = router_linear(xd, wd)
    _near(y, x, w.t(), h)
    with torch.no_grad():
        assert torch.equal(router_linear(xd, wd), y)
    y.backward(d.cuda())
    _near(wd.grad, d.t(), x, t)
    _near(xd.grad, d, w, e)


def test_fp32_logits_and_other_kinds_of_input():
    from qwen3_moe_fused import _lib

    x, w = (torch.randn(s, generator=gen(s[0])).to(torch.bfloat16) for s in ((530, 256), (72, 256)))
    xd, wd = x.cuda(), w.cuda()
    out = torch.empty((530, 72), device="cuda")
    for t in (530, 40):
        _lib.check(_lib.lib().mfl_router_fwd(xd.data_ptr(), wd.data_ptr(), out.data_ptr(), t, 256, 72, _lib.F32, _lib.stream()),
                   "mfl_router_fwd")
        _near(out[:t], x[:t], w.t(), 256, 2.0 ** -23)
    assert router_linear(xd.float(), wd) is None and router_linear(xd[:, :64], wd[:, :64]) is None
    gate = Qwen3MoeFusedRouter(256, 72, bias=False).cuda()
    z = torch.randn((3, 5, 256)).cuda()
    assert torch.equal(gate(z), torch.nn.functional.linear(z, gate.weight))


def test_router_gradients_of_gradients_and_forward_mode():
    """What the stock projection takes: a penalty on its gradients, and tangents."""
    t, h, e = 600, 128, 16
    x, w, d = (torch.randn(s, generator=gen(7)).to(torch.bfloat16).cuda() for s in ((t, h), (e, h), (t, e)))
    gate = Qwen3MoeFusedRouter(h, e, bias=False).to("cuda", torch.bfloat16)
    got = []
    for f in (gate, lambda z: torch.nn.functional.linear(z, gate.weight)):
        xr = x.clone().requires_grad_()
        gate.weight.data.copy_(w)
        (dx,) = torch.autograd.grad((f(xr) * d).sum(), xr, create_graph=True)
        got.append(torch.autograd.grad(dx.float().square().sum(), gate.weight)[0])
        with torch.autograd.forward_ad.dual_level(), torch.no_grad():
            dual = f(torch.autograd.forward_ad.make_dual(x, x))
            got.append(torch.autograd.forward_ad.unpack_dual(dual).tangent)
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])


def test_router_weight_gradient_keeps_an_infinity_of_the_last_token():
    t, h, e = 513, 128, 16
    x, d = torch.ones((t, h)).to(torch.bfloat16).cuda(), torch.ones((t, e)).to(torch.bfloat16).cuda()
    w = torch.zeros((e, h), device="cuda", dtype=torch.bfloat16).requires_grad_()
    x[-1, 5] = float("inf")
    router_linear(x, w).backward(d)
    assert torch.isinf(w.grad[:, 5]).all() and (torch.cat((w.grad[:, :5], w.grad[:, 6:]), 1) == 512).all()  # 513 in bf16


@pytest.mark.parametrize("grad", [False, True])
def test_router_compiles_as_a_whole(grad):
    gate = Qwen3MoeFusedRouter(128, 16, bias=False).to("cuda", torch.bfloat16)
    x = torch.randn((40, 128), generator=gen(1)).to(torch.bfloat16).cuda().requires_grad_(grad)
    with torch.set_grad_enabled(grad):
        out = torch.compile(gate, fullgraph=True, backend="eager")(x)
        assert torch.equal(out, torch.nn.functional.linear(x, gate.weight))


def test_block_compiles_around_its_kernels():
    from test_gpu_block_call import _block

    blk, dtype = _block(8, 2, 64, 64, "bf16", 3)
    x = torch.randn((1, 40, 64), generator=gen(1)).to(dtype).cuda()
    with torch.no_grad():
        want = blk(x)
        got = torch.compile(blk, backend="eager")(x)
    for a, b in zip(got, want):
        assert (a.float() - b.float()).abs().max() <= 2e-2 * b.float().abs().max()


def test_router_gradients_several_at_once():
    x, w, d = (torch.randn(s, generator=gen(5)).to(torch.bfloat16).cuda() for s in ((600, 128), (16, 128), (2, 600, 16)))
    x.requires_grad_(), w.requires_grad_()
    got = torch.autograd.grad(router_linear(x, w), (x, w), d, is_grads_batched=True)
    for i in range(2):
        _near(got[0][i], d[i].cpu(), w.detach().cpu(), 16)
        _near(got[1][i], d[i].t().cpu(), x.detach().cpu(), 600)


@pytest.mark.parametrize("t,h,e", [(511, 640, 264), (33, 7168, 40), (530, 64, 520)])
def test_projection_kernel_beyond_where_the_module_takes_it(t, h, e):
    from qwen3_moe_fused import _lib

    x, w = (torch.randn(s, generator=gen(t)).to(torch.bfloat16) for s in ((t, h), (e, h)))
    xd, wd, out = x.cuda(), w.cuda(), torch.empty((t, e), dtype=torch.bfloat16, device="cuda")
    _lib.check(_lib.lib().mfl_router_fwd(xd.data_ptr(), wd.data_ptr(), out.data_ptr(), t, h, e, _lib.BF16, _lib.stream()),
               "mfl_router_fwd")
    _near(out, x, w.t(), h)
