"""Shared helpers of the parity tests: seeded inputs, routing draws, error metrics."""
from __future__ import annotations

import re
import warnings

import numpy as np
import torch

import oracle

# bf16 GEMM tolerance: the reference's own criterion, allclose(rtol=1e-2, atol=1e-2)
# (test_moe_fused_linear.py:34-36,52), plus max|a-b| / max|ref| <= 1e-2.
BF16_RTOL = 1e-2
BF16_ATOL = 1e-2


def gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    return g


def randn(shape, g, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, dtype=torch.float32) * scale).to(dtype)


def to_np32(t: torch.Tensor) -> np.ndarray:
    return t.detach().float().cpu().numpy()


def m_sizes_uniform(rows: int, E: int, g) -> torch.Tensor:
    """Per-expert counts of `rows` rows drawn uniformly over E experts (sorted batch)."""
    sel = torch.randint(0, E, (rows,), generator=g)
    return torch.bincount(sel, minlength=E).to(torch.int32)


def topk_routing(T: int, E: int, k: int, g, bias=None):
    """softmax -> top-k routing of T tokens; returns (sel (T*k,) int64, m_sizes int32)."""
    logits = torch.randn((T, E), generator=g)
    if bias is not None:
        logits = logits + bias
    sel = torch.topk(torch.softmax(logits, dim=-1), k, dim=-1).indices.reshape(-1)
    return sel, torch.bincount(sel, minlength=E).to(torch.int32)


def zipf_bias(E: int, s: float, g) -> torch.Tensor:
    """log-popularity of experts, p_e ~ rank^-s under a seeded random rank permutation."""
    ranks = torch.randperm(E, generator=g).float() + 1.0
    p = ranks.pow(-s)
    return (p / p.sum()).log()


def check_close(actual: torch.Tensor, expect: np.ndarray, rtol=BF16_RTOL, atol=BF16_ATOL, what=""):
    a = to_np32(actual).astype(np.float64)
    e = np.asarray(expect, dtype=np.float64)
    assert a.shape == e.shape, f"{what}: shape {a.shape} vs {e.shape}"
    assert np.isfinite(a).all(), f"{what}: non-finite values"
    diff = np.abs(a - e)
    scale = max(np.abs(e).max(), 1e-30) if e.size else 1.0
    norm_max = diff.max() / scale if e.size else 0.0
    ok = (diff <= atol + rtol * np.abs(e)).all()
    assert ok and norm_max <= rtol, (
        f"{what}: allclose={ok} normalised max err={norm_max:.3e} max abs err={diff.max():.3e} (ref max {scale:.3e})")
    return norm_max


def unit_scale_atol(expect: np.ndarray, atol=BF16_ATOL) -> float:
    """The absolute tolerance of the reference's tests, carried over to outputs that are not of unit scale.

    The reference draws weights with standard deviation 1 / sqrt(K) so that outputs have unit scale and
    atol = 1e-2 is one percent of it (test_moe_fused_linear.py:33-38).  For outputs of another scale the same
    one percent is atol * std(expect).  Used where the kernel does not reproduce the reference's rounded
    weights bit for bit: the decode-size NF4 kernel multiplies bf16(code) and applies absmax to a
    quantisation block's partial sum, the reference multiplies bf16(code * absmax); the two differ by
    rounding noise of a bf16 ulp per weight, which a sum over K elements turns into about 1e-3 of the
    output scale."""
    return atol * max(1.0, float(np.asarray(expect, dtype=np.float64).std()))


def oracle_rows(x: torch.Tensor, w: torch.Tensor, sel: np.ndarray, rows: np.ndarray) -> np.ndarray:
    """Oracle forward for a subset of rows (rows are independent)."""
    return oracle.linear_fwd(to_np32(x[rows]), to_np32(w), sel[rows])


_TILED = re.compile(r"gemm_(pipe|wide)_kernel(I|<)(.*)")


def tiles_of(fn):
    """``(fn(), tiles)`` with the tiles that the pipelined and four-wave products launched by ``fn`` ran on, from the names
    of their kernels: a set of ``(kernel, rows, columns, product, packed, fusion)``, kernel "pipe" or "wide", product 0
    forward, 1 input gradient, 2 weight gradient, fusion as the pipelined kernel's template has it (0 none, 1 gated, 2 thin
    last term, 3 both, 4 gated unit's backward).  None where the tracer gave no kernels at all (another tool may hold it)."""
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        out = fn()
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA]
    if not names:
        warnings.warn("no kernel names from the tracer: the tiles are not checked")
        return out, None
    found = set()
    for name in names:
        m = _TILED.search(name)
        if m is None:
            continue
        if m[2] == "I":  # mangled: Li<number>E, Lb<0 or 1>E
            args = [int(v) for v in re.findall(r"L[ib](\d+)E", m[3])]
        else:
            args = [int({"true": 1, "false": 0}.get(v, v)) for v in re.findall(r"true|false|\b\d+\b", m[3].split(">")[0])]
        if m[1] == "pipe":
            mb, nb, _, _, _, _, mode, packed, fuse = args[:9]
        else:
            mode, mb, nb, _, _, thin = args[:6]
            packed, fuse = 0, 2 * thin
        found.add((m[1], 32 * mb, 32 * nb, mode, bool(packed), fuse))
    return out, found


def check_tiles(fn, *expect):
    """``fn()``, which has to run on exactly these tiles (see ``tiles_of``)."""
    out, found = tiles_of(fn)
    assert found is None or found == set(expect), f"ran on {sorted(found)}, expected {sorted(expect)}"
    return out
