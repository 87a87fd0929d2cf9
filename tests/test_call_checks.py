"""What the wrappers refuse or leave to the stock operators, on the CPU: the tensors claim to be on the GPU and the
library is a stand-in, so that a call which would hand raw pointers to a kernel shows itself instead."""
import pytest
import torch

from qwen3_moe_fused import _lib
from qwen3_moe_fused.kernels import routing


class LibraryCalled(Exception):
    pass


class _StandIn:
    def __getattr__(self, name):
        raise LibraryCalled(name)


@pytest.fixture
def no_kernels(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "lib", lambda: _StandIn())
    monkeypatch.setattr(_lib, "stream", lambda: 0)


def _bf16(*shape):
    return torch.ones(shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("width", [64, 192])
def test_router_refuses_rows_of_another_width(no_kernels, width, grad):
    w = _bf16(8, 128).requires_grad_(grad)
    with pytest.raises(LibraryCalled):  # the stand-in is where a call of the right width goes
        routing.router_linear(_bf16(4, 128), w)
    x = _bf16(4, width)
    with pytest.raises(RuntimeError, match="cannot be multiplied"):
        out = routing.router_linear(x, w)
        torch.nn.functional.linear(x, w) if out is None else out


def _dense(t=6, e=4, h=32, i=16, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(1)
    return [torch.randn(s, generator=g).to(dtype) for s in ((t, h), (t, e), (e, i, h), (e, i, h), (e, h, i))]


# position of the tensor that does not fit (tokens, logits, gate, up, down) and what stands there instead
MISFITS = [(0, (6, 16)), (0, (6, 48)), (0, (5, 32)), (1, (6, 3)), (1, (6, 5)), (1, (7, 4)), (2, (3, 16, 32)), (2, (4, 8, 32)),
           (3, (4, 8, 32)), (3, (4, 24, 32)), (3, (5, 16, 32)), (4, (4, 16, 32)), (4, (3, 32, 16)), (4, (4, 40, 16)),
           (2, (64, 32))]


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("which,shape", MISFITS)
def test_block_call_refuses_operands_that_do_not_fit(no_kernels, which, shape, grad):
    from qwen3_moe_fused.fused_mlp import moe_block

    args = _dense()
    with pytest.raises(LibraryCalled):
        moe_block(*args, 2, True)
    args[which] = torch.zeros(shape, dtype=torch.bfloat16)
    args[4].requires_grad_(grad)
    with pytest.raises(AssertionError):
        moe_block(*args, 2, True)


def _strided(t):
    return torch.empty((*t.shape[:-1], t.shape[-1] + 1), dtype=t.dtype)[..., :-1]


@pytest.mark.parametrize("which", range(5))
@pytest.mark.parametrize("how", [_strided, torch.Tensor.double, lambda t: t.to("meta")], ids=["strided", "type", "device"])
def test_block_call_refuses_strides_types_and_devices(no_kernels, which, how):
    from qwen3_moe_fused.fused_mlp import moe_block

    args = _dense()
    args[which] = how(args[which])
    with pytest.raises((AssertionError, TypeError)):
        moe_block(*args, 2, True)


@pytest.mark.parametrize("e", [3, 5])
def test_block_call_on_packed_weights_refuses_logits_of_other_experts(no_kernels, e):
    from qwen3_moe_fused import fused_mlp

    tokens, _, gate, up, down = _packed_block()
    with pytest.raises(AssertionError):
        fused_mlp.moe_block_4bit(tokens, torch.zeros((6, e), dtype=torch.bfloat16), gate, up, down, 2, True)
    with pytest.raises(LibraryCalled):
        fused_mlp.moe_block_4bit(tokens, torch.zeros((6, 4), dtype=torch.bfloat16), gate, up, down, 2, True)


def _packed_block(t=6, e=4, h=128, i=64):
    from qwen3_moe_fused.quantize.layer import Nf4Params
    from qwen3_moe_fused.quantize.nf4 import BlockwiseState, Nf4QuantState, code_of

    def packed(n, k):
        state = Nf4QuantState(absmax=torch.ones(e * n * k // 64, dtype=torch.uint8), shape=(e, n, k), code=code_of("nf4", "cpu"),
                              blocksize=64, quant_type="nf4", dtype=torch.bfloat16, offset=torch.zeros(()),
                              state2=BlockwiseState(absmax=torch.ones(e * n * k // 64 // 4), code=torch.zeros(256), blocksize=4))
        return Nf4Params(torch.zeros((e * n * k // 2, 1), dtype=torch.uint8), quant_state=state)

    return _bf16(t, h), None, packed(i, h), packed(i, h), packed(h, i)


def test_nothing_on_the_host_reaches_the_block_kernels(monkeypatch):
    """A block on the CPU was refused by the checks of the separate steps: as one call it is as well."""
    from types import SimpleNamespace

    from qwen3_moe_fused.modular_qwen3_moe_fused import Qwen3MoeFusedSparseMoeBlock

    monkeypatch.setattr(_lib, "lib", lambda: _StandIn())
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    block = Qwen3MoeFusedSparseMoeBlock(SimpleNamespace(
        num_experts=4, num_experts_per_tok=2, norm_topk_prob=True, hidden_size=32, moe_intermediate_size=16,
        hidden_act="silu"))
    with pytest.raises(AssertionError):
        block(torch.zeros((1, 3, 32)))
    from qwen3_moe_fused.fused_mlp import moe_block_4bit

    tokens, _, gate, up, down = _packed_block()
    with pytest.raises(AssertionError):
        moe_block_4bit(tokens, torch.zeros((6, 4), dtype=torch.bfloat16), gate, up, down, 2, True)


class _Recorder:
    """Stands for the library: notes the packed matrices that a product is given and answers as told."""

    def __init__(self, answers):
        self.seen, self.answers = [], answers

    def __getattr__(self, name):
        def call(*args):
            self.seen.append((name, [(a.absmax_u8 is not None, a.blocksize2) for a in args if isinstance(a, _lib.Nf4Weight)]))
            return self.answers.get(name, 0)

        return call


def _with_blocksize2(w, blocksize2):
    st = w.quant_state
    st.state2.blocksize = blocksize2
    st.state2.absmax = torch.ones(-(-st.absmax.numel() // blocksize2))
    return w


# A second level in blocks that are not a power of two, or of one scale each, has no kernel of its own: the scales are
# written out first, as they were for every product.
@pytest.mark.parametrize("blocksize2", [1, 3, 100])
def test_other_second_level_blocks_are_written_out(monkeypatch, blocksize2):
    from qwen3_moe_fused import fused_mlp
    from qwen3_moe_fused.grouped_gemm import forward_4bit, fused

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    tokens, _, gate, up, down = (t if i < 2 else _with_blocksize2(t, blocksize2) for i, t in enumerate(_packed_block()))
    sizes, rows = torch.full((4,), 3, dtype=torch.int32), torch.zeros(12, dtype=torch.int32)
    products = {
        "mfl_gemm_fwd_nf4_packed": [
            lambda: forward_4bit.grouped_gemm_forward_4bit(_bf16(12, 128), gate, gate.quant_state, sizes),
            lambda: fused.grouped_gemm_forward_4bit_gathered(tokens, rows, 2, gate, gate.quant_state, sizes)],
        "mfl_glu_fwd_nf4_packed": [
            lambda: fused.grouped_glu_forward_4bit(tokens, gate, gate.quant_state, up, up.quant_state, sizes, rows, 2)]}
    for name, calls in products.items():
        for call in calls:
            lib = _Recorder({})
            monkeypatch.setattr(_lib, "lib", lambda: lib)
            call()
            given = [w for n, w in lib.seen if n == name]
            assert given and not any(nested for ws in given for nested, _ in ws)
            assert any(n == "mfl_dequant_blockwise_u8" for n, _ in lib.seen)
    lib = _Recorder({})
    fused_mlp.moe_block_4bit(tokens, torch.zeros((6, 4), dtype=torch.bfloat16), gate, up, down, 2, True)
    names = [n for n, _ in lib.seen]
    assert names[-1] == "mfl_moe_block_fwd" and names.count("mfl_dequant_blockwise_u8") == 3


@pytest.mark.parametrize("nested", [False, True])
def test_strided_scales_are_taken(monkeypatch, nested):
    """A state's scales may lie apart (a view of more): they are made contiguous for the kernels."""
    from qwen3_moe_fused.grouped_gemm import forward_4bit

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    tokens, _, gate, _, _ = _packed_block()
    st = gate.quant_state
    if not nested:
        st.absmax, st.state2, st.offset = torch.ones(st.absmax.numel()), None, None
    assert st.nested == nested
    st.absmax = torch.stack((st.absmax, st.absmax), dim=1)[:, 0]
    assert not st.absmax.is_contiguous()
    lib = _Recorder({})
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    forward_4bit.grouped_gemm_forward_4bit(tokens, gate, st, torch.tensor([6, 0, 0, 0], dtype=torch.int32))
    assert lib.seen[-1] == ("mfl_gemm_fwd_nf4_packed", [(nested, 4 if nested else 0)])


@pytest.mark.parametrize("offset", [None, 0.25, torch.tensor(0.25), torch.tensor([0.25], dtype=torch.float64)])
def test_an_offset_of_any_kind_is_made_on_the_device(monkeypatch, offset):
    """None and plain numbers become a one-element tensor by a fill, which a stream capture takes; a copy from the host
    (what ``torch.tensor(value, device=...)`` does) it refuses."""
    from qwen3_moe_fused.quantize import nf4

    state = _packed_block()[2].quant_state
    state.offset = offset

    def from_host(*args, **kwargs):
        raise AssertionError("a copy from the host")

    monkeypatch.setattr(torch, "tensor", from_host)
    off = nf4._second_level(state)[4]
    assert off.numel() == 1 and off.dtype == torch.float32 and float(off) == (0.0 if offset is None else 0.25)


def _lora_args(rows=4096, e=2, h=16, m=16, r=8, rb=None):
    """Operands of the fast-LoRA function; ``rb``: another rank in the B matrices of gate and up."""
    a, b = (_bf16(e, r, h), _bf16(e, m, rb or r))
    return [_bf16(rows, h), _bf16(e, m, h), None, a, b, 1.0, _bf16(e, m, h), None, a.clone(), b.clone(), 1.0, _bf16(e, h, m), None,
            _bf16(e, r, m), _bf16(e, h, r), 1.0, torch.tensor([rows - 1, 1], dtype=torch.int32)]


@pytest.mark.parametrize("rb", [4, 12, 16, 24])
def test_thin_matrices_of_unequal_rank_are_refused(monkeypatch, rb):
    from qwen3_moe_fused.kernels.fast_lora import fast_lora

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    for args, fits in ((_lora_args(), True), (_lora_args(rb=rb), False)):
        lib = _Recorder({})
        monkeypatch.setattr(_lib, "lib", lambda: lib)
        if fits:
            fast_lora(*args)
            assert lib.seen[0][0] == "mfl_copy_blocks"
        else:
            with pytest.raises(AssertionError):
                fast_lora(*args)
            assert not lib.seen


@pytest.mark.parametrize("elsewhere", [(), (3, 8), (4, 9), (3,), (8,), (9,)])
def test_thin_matrices_on_another_device_never_reach_the_copies(monkeypatch, elsewhere):
    """Operands on the host, or on another device than the rows, are refused by the products; the copies that join the
    thin matrices come before those.  (): all of them on the host."""
    from qwen3_moe_fused.kernels.fast_lora import fast_lora

    if elsewhere:
        monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    lib = _Recorder({})
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    with pytest.raises((AssertionError, RuntimeError)):
        fast_lora(*(t.to("meta") if i in elsewhere else t for i, t in enumerate(_lora_args())))
    assert not lib.seen


def _double_quantised(device, numel=4 * 16 * 16 // 64, blocksize2=4):
    from qwen3_moe_fused.quantize.nf4 import BlockwiseState, Nf4QuantState, code_of

    return Nf4QuantState(absmax=torch.ones(numel, dtype=torch.uint8, device=device), shape=(2, 16, 16),
                         code=code_of("nf4", device), blocksize=64, quant_type="nf4", dtype=torch.bfloat16,
                         offset=torch.zeros((), device=device),
                         state2=BlockwiseState(absmax=torch.ones(-(-numel // blocksize2), device=device),
                                               code=torch.zeros(256, device=device), blocksize=blocksize2))


@pytest.mark.parametrize("states_on,rows_on_gpu", [("cpu", False), ("meta", False), ("meta", True)])
def test_scales_on_another_device_than_the_rows_are_not_written_out(monkeypatch, states_on, rows_on_gpu):
    """The scales are written out before the products, whose checks refuse weights that are not on the rows' GPU: with states
    elsewhere (an offloaded layer), or with everything on the host, no kernel sees an address."""
    from qwen3_moe_fused.kernels.fast_lora import fast_lora

    if rows_on_gpu:
        monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    lib = _Recorder({})
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    args = _lora_args(rows=64)
    for i in (1, 6, 11):
        args[i], args[i + 1] = torch.zeros((2 * 16 * 16 // 2, 1), dtype=torch.uint8), _double_quantised(states_on, 2 * 16 * 16 // 64)
    with pytest.raises((AssertionError, RuntimeError)):
        fast_lora(*args)
    assert not any(name in ("mfl_nf4_write_out_scales", "mfl_nf4_unnest_absmax") for name, _ in lib.seen)


def test_scales_are_written_out_under_inference_mode(monkeypatch):
    """A tensor made under inference mode has no version to ask for."""
    from qwen3_moe_fused.quantize.nf4 import tiled_absmax, write_out_scales

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    lib = _Recorder({})
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    state = _double_quantised("cpu", 2 * 16 * 16 // 64)
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            out, = write_out_scales(torch.zeros(2, 16), state)
            assert out is not state and not out.nested and tiled_absmax(out, out.absmax, 2) is None
    assert [name for name, _ in lib.seen] == ["mfl_nf4_write_out_scales"] * 2


def test_a_state_that_several_matrices_share_is_written_out_once(monkeypatch):
    """The room for a state's scales is kept until the launch: a second piece for the same state would replace the first one,
    whose memory the next state could get while the kernel still writes both."""
    from qwen3_moe_fused.quantize.nf4 import write_out_scales

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    jobs = []

    class Library:
        def mfl_nf4_write_out_scales(self, weights, counts, ptrs, n, stream):
            jobs.append([(counts[i], ptrs[i]) for i in range(n)])
            return 0

    monkeypatch.setattr(_lib, "lib", lambda: Library())
    a, b = _double_quantised("cpu", 4096), _double_quantised("cpu", 4096)
    outs = write_out_scales(torch.zeros(2, 16), a, a, b)
    assert outs[0] is outs[1] and outs[2] is not outs[0]
    assert jobs == [[(4096, outs[0].absmax.data_ptr()), (4096, outs[2].absmax.data_ptr())]]
    assert outs[0].absmax.data_ptr() != outs[2].absmax.data_ptr()


@pytest.mark.parametrize("h", [64, 96, 192, 224])
def test_packed_gate_and_up_in_one_launch_for_whole_reduction_steps(monkeypatch, h):
    """For other hidden sizes there is no such kernel, and the separate products take each adapter's own rank."""
    from qwen3_moe_fused.kernels.fast_lora import fast_lora
    from qwen3_moe_fused.quantize.nf4 import Nf4QuantState, code_of

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    names, ranks = [], []

    class Library:
        def __getattr__(self, name):
            def call(*args):
                names.append(name)
                if name == "mfl_gemm_fwd_nf4_lora":
                    ranks.append(args[7])
                return 0

            return call

    monkeypatch.setattr(_lib, "lib", lambda: Library())
    args = _lora_args(h=h, m=64, r=8)
    for i, shape in ((1, (2, 64, h)), (6, (2, 64, h)), (11, (2, h, 64))):
        args[i] = torch.zeros((2 * 64 * h // 2, 1), dtype=torch.uint8)
        args[i + 1] = Nf4QuantState(absmax=torch.ones(2 * 64 * h // 32), shape=shape, code=code_of("nf4", "cpu"), blocksize=32,
                                    quant_type="nf4", dtype=torch.bfloat16)
    fast_lora(*args)
    assert names.count("mfl_glu_fwd_nf4_lora") == (h % 64 == 0)
    assert names.count("mfl_gemm_fwd_nf4_lora") == (1 if h % 64 == 0 else 3) and set(ranks) == {8}


def _router_and_rows():
    from qwen3_moe_fused.modular_qwen3_moe_fused import Qwen3MoeFusedRouter

    return Qwen3MoeFusedRouter(64, 8, bias=False), torch.randn(3, 64)


def _compiled(m, x):
    return torch.compile(m, fullgraph=True, backend="eager")


# the router is a linear layer to whoever records or compiles it
@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("how", [lambda m, x: torch.jit.script(m), lambda m, x: torch.jit.trace(m, (x,)), _compiled,
                                 lambda m, x: torch.fx.symbolic_trace(m),
                                 lambda m, x: torch.export.export(m, (x,)).module(),
                                 lambda m, x: torch.export.export(m, (x,), strict=True).module()],
                         ids=["script", "trace", "compile", "fx", "export", "export-strict"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_router_is_recorded_as_a_linear_layer(how, dtype):
    m, x = _router_and_rows()
    m, x = m.to(dtype), x.to(dtype)
    assert torch.equal(how(m, x)(x), torch.nn.functional.linear(x, m.weight))


@pytest.mark.parametrize("tokens", [4, 600])
def test_router_gradients_batched_and_under_modes_are_the_stock_products(monkeypatch, tokens):
    """Several gradients at once (``is_grads_batched``, vectorised Jacobians) run the backward on batched tensors, which have
    no address; an operator counter around the backward sees its products."""
    from torch.utils.flop_counter import FlopCounterMode

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "stream", lambda: 0)
    monkeypatch.setattr(routing, "_router_logits", torch.nn.functional.linear)
    lib = _Recorder({})
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    g = torch.Generator().manual_seed(tokens)
    x, w, d = (torch.randn(s, generator=g).to(torch.bfloat16) for s in ((tokens, 64), (8, 64), (3, tokens, 8)))
    x.requires_grad_(), w.requires_grad_()
    y = routing.router_linear(x, w)
    assert type(y.grad_fn).__name__ == "_RouterLinearBackward"
    got = torch.autograd.grad(y, (x, w), d, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for a, b in zip(got, torch.autograd.grad(torch.nn.functional.linear(x, w), (x, w), d[i])):
            assert torch.allclose(a[i].float(), b.float(), rtol=2 ** -7, atol=1e-2)
    with FlopCounterMode(display=False) as count:
        torch.autograd.grad(y, (x, w), d[0])
    assert count.get_total_flops() == 2 * 2 * tokens * 64 * 8 and not lib.seen


def _small_block(kind="bf16"):
    from types import SimpleNamespace

    from qwen3_moe_fused.modular_qwen3_moe_fused import Qwen3MoeFusedSparseMoeBlock
    from qwen3_moe_fused.quantize.layer import MoeFusedLinear4bit

    block = Qwen3MoeFusedSparseMoeBlock(SimpleNamespace(
        num_experts=4, num_experts_per_tok=2, norm_topk_prob=True, hidden_size=128, moe_intermediate_size=64,
        hidden_act="silu")).to(torch.bfloat16)
    if kind == "nf4":
        for name, w in zip(("gate_proj", "up_proj", "down_proj"), _packed_block()[2:]):
            proj = MoeFusedLinear4bit(*w.quant_state.shape[:0:-1], 4, device="meta")
            proj._parameters["weight"] = w
            setattr(block, name, proj)
    return block


@pytest.mark.parametrize("kind", ["bf16", "nf4"])
@pytest.mark.parametrize("how", ["class", "instance", "hook"])
def test_block_call_steps_aside_for_replaced_forwards(no_kernels, monkeypatch, kind, how):
    block = _small_block(kind)
    tokens, logits = _bf16(3, 128), _bf16(3, 4)
    with torch.no_grad():
        with pytest.raises(LibraryCalled):
            block._one_call(tokens, logits)
        if how == "class":
            plain = type(block.down_proj).forward
            monkeypatch.setattr(type(block.down_proj), "forward", lambda self, *a: plain(self, *a))
        elif how == "instance":
            block.down_proj.forward = block.down_proj.forward
        else:
            block.down_proj.register_forward_hook(lambda m, a, o: None)
        assert block._one_call(tokens, logits) is None


def test_router_is_seen_by_function_modes(no_kernels):
    from torch.overrides import TorchFunctionMode

    class Seen(TorchFunctionMode):
        names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    gate, x = _router_and_rows()
    gate, x = gate.to(torch.bfloat16), x.to(torch.bfloat16)
    with torch.no_grad():
        with pytest.raises(LibraryCalled):
            gate(x)
        with torch.device("cpu"), pytest.raises(LibraryCalled):  # a default device watches nothing
            gate(x)
        with Seen(), torch.device("cpu"):
            gate(x)
    assert "linear" in Seen.names


# tokens of 8 selections each, 128 experts, hidden 2048, intermediate 768: the gated product reads 8-bit scales up to 384
# rows per expert, the plain one up to 128; with K = 96, or second-level blocks shorter than a row, neither does
@pytest.mark.parametrize("tokens,inter,blocksize2,slots", [(1, 768, 256, 0), (256, 768, 256, 0), (2048, 768, 256, 0),
                                                           (2049, 768, 256, 1), (6144, 768, 256, 1), (6145, 768, 256, 2),
                                                           (1, 96, 256, 1), (1, 768, 16, 2)])
def test_block_workspace_has_room_for_written_out_scales_only_where_they_are(tokens, inter, blocksize2, slots):
    import ctypes

    def size(nested):
        at = 1 << 20  # (an address that is compared with alignments, never followed)
        w = _lib.Nf4Weight(at, at, None if nested else at, None, at if nested else None, at, at, at, 64, blocksize2)
        p = ctypes.pointer(w)
        b = _lib.MoeBlock(at, at, None, None, None, p, p, p, tokens, 128, 8, 2048, inter, 1, _lib.BF16, _lib.BF16, 0)
        return _lib.lib().mfl_moe_block_workspace(b)

    assert size(True) - size(False) == slots * 128 * 2048 * inter // 64 * 4


def test_block_workspace_on_packed_weights_never_holds_the_two_products():
    """More than 512 experts: the dense form keeps gate's and up's products for a separate SiLU-mul, the packed kernels do
    not need them."""
    import ctypes

    def size(experts):
        at = 1 << 20
        p = ctypes.pointer(_lib.Nf4Weight(at, at, at, None, None, None, None, None, 64, 0))
        b = _lib.MoeBlock(at, at, None, None, None, p, p, p, 16, experts, 8, 512, 256, 1, _lib.BF16, _lib.BF16, 0)
        return _lib.lib().mfl_moe_block_workspace(b)

    assert size(513) - size(512) < 16 * 8 * 256 * 2


# (tokens, hidden, experts): where the router's own kernel takes the projection, and where the stock product is ahead of it
@pytest.mark.parametrize("t,h,e,own", [(1, 64, 1, True), (512, 4096, 128, True), (513, 2048, 8, False), (1, 5184, 8, False),
                                       (512, 64, 256, True), (512, 64, 257, False), (512, 2048, 256, True), (512, 2112, 256, False),
                                       (512, 4096, 129, False), (192, 5120, 272, True), (193, 5120, 272, False)])
def test_router_projection_takes_its_own_kernel_where_that_is_ahead(no_kernels, t, h, e, own):
    if own:
        with pytest.raises(LibraryCalled):
            routing.router_linear(_bf16(t, h), _bf16(e, h))
    else:
        assert routing.router_linear(_bf16(t, h), _bf16(e, h)).shape == (t, e)


@pytest.mark.parametrize("t,h,e,own", [(512, 4096, 512, True), (512, 4104, 512, False), (511, 64, 8, False)])
def test_router_weight_gradient_takes_its_own_kernel_where_that_is_ahead(no_kernels, monkeypatch, t, h, e, own):
    monkeypatch.setattr(routing, "_router_logits", torch.nn.functional.linear)
    w = _bf16(e, h).requires_grad_()
    y = routing.router_linear(_bf16(t, h), w)
    if own:
        with pytest.raises(LibraryCalled):
            y.backward(_bf16(t, e))
    else:
        y.backward(_bf16(t, e))
        assert w.grad.shape == (e, h)


@pytest.mark.parametrize("tokens,grad,frozen,own", [(1, True, True, True), (512, False, False, True), (513, True, False, False),
                                                    (2047, True, False, False), (2048, True, False, True), (2048, True, True, False),
                                                    (2048, False, False, False)])
def test_router_module_is_the_stock_node_where_no_kernel_of_its_own_runs(monkeypatch, tokens, grad, frozen, own):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    seen = []
    from qwen3_moe_fused import modular_qwen3_moe_fused as mod

    monkeypatch.setattr(mod, "router_linear", lambda x, w: seen.append(1))
    gate = mod.Qwen3MoeFusedRouter(64, 8, bias=False).to(torch.bfloat16)
    gate.weight.requires_grad_(not frozen)
    with torch.set_grad_enabled(grad):
        gate(_bf16(tokens, 64))
    assert bool(seen) == own
