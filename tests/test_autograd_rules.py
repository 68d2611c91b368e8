"""CPU tests of the ops' autograd rules, on meta tensors (shapes only, nothing is launched).

What has no formula must refuse a gradient: dropping it gives a caller wrong
gradients without an error.
"""

from __future__ import annotations

import os
import subprocess
import sys

import pytest
import torch

BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def ops(mta):
    mta._native.load()
    return torch.ops.mega_trading_amd


def meta(*shape, dtype=torch.float32, grad=True):
    return torch.empty(*shape, dtype=dtype, device="meta", requires_grad=grad)


def tables():
    return meta(8, 16, grad=False), meta(8, 16, grad=False)


def heads(n, t=8):
    return meta(2, n, t, 32, dtype=BF16)


NO_FORMULA = {
    "gqa_attn_decode": lambda: (heads(4, 1), heads(2), heads(2), 5, 0.2),
    "gqa_attn_decode_dev": lambda: (heads(4, 1), heads(2), heads(2), torch.ones(1, dtype=torch.int32, device="meta"), 0.2),
    "decode_rope_append": lambda: (heads(4, 1), heads(2, 1), heads(2, 1), *tables(), 3, None,
                                   heads(2).detach(), heads(2).detach()),
    "gqa_attn_decode_append": lambda: (heads(4, 1), heads(2, 1), heads(2, 1), *tables(), 3, None, 4, None,
                                       heads(2).detach(), heads(2).detach(), 0.2),
    "linear_rows": lambda: (meta(4, 128), [meta(8, 128), meta(16, 128)]),
    "linear_rows_gate": lambda: (meta(4, 128), meta(8, 128), meta(8, 128)),
    "rms_norm_bwd": lambda: (meta(4, 16), meta(16), meta(4), meta(4, 16)),
    "swiglu_bwd": lambda: (meta(4, 16), meta(4, 16), meta(4, 16)),
    "scale_pair": lambda: (meta(4, 16), meta(16), torch.zeros((), device="meta", requires_grad=True)),
}
SECOND_ORDER = {
    "gqa_attn_fwd": lambda: (heads(4), heads(2), heads(2), 0.2),
    "gqa_rope_attn_fwd": lambda: (heads(4), heads(2), heads(2), *tables(), 0.2),
    "rms_norm_fwd": lambda: (meta(4, 16), meta(16), 1e-5),
    "add_rms_norm_fwd": lambda: (meta(4, 16), meta(4, 16), meta(16), 1e-5),
    "rms_norm_fwd_mixed": lambda: (meta(4, 16), meta(16), 1e-5, 0),
    "swiglu_fwd": lambda: (meta(4, 16), meta(4, 16)),
    "swiglu_packed_fwd": lambda: (meta(4, 32),),
}


def call(op, args):
    out = op(*args)
    outs = out if isinstance(out, (tuple, list)) else (out,)
    flat = [y for x in args for y in (x if isinstance(x, list) else [x])]
    return outs, [x for x in flat if isinstance(x, torch.Tensor) and x.requires_grad]


@pytest.mark.parametrize("name", sorted(NO_FORMULA))
def test_a_gradient_through_an_op_without_a_formula_is_refused(ops, name):
    outs, leaves = call(getattr(ops, name), NO_FORMULA[name]())
    for out in outs:
        assert out.requires_grad
        with pytest.raises(RuntimeError, match="no autograd formula"):
            torch.autograd.grad(out, leaves, torch.ones_like(out), allow_unused=True, retain_graph=True)
    with torch.no_grad():
        assert not call(getattr(ops, name), NO_FORMULA[name]())[0][0].requires_grad


@pytest.mark.parametrize("name", sorted(SECOND_ORDER))
def test_a_second_order_gradient_is_refused(ops, name):
    outs, leaves = call(getattr(ops, name), SECOND_ORDER[name]())
    first = torch.autograd.grad(outs[-2] if name == "add_rms_norm_fwd" else outs[0], leaves, torch.ones_like(outs[0]),
                                create_graph=True)
    for g in first:
        with pytest.raises(RuntimeError, match="no autograd formula"):
            torch.autograd.grad(g, leaves, torch.ones_like(g), allow_unused=True, retain_graph=True)


def test_the_mixed_residual_norm_refuses_a_second_order_gradient(ops):
    x, r, w = meta(4, 16, dtype=BF16), meta(4, 16), meta(16)
    _res, y, _rstd = ops.add_rms_norm_fwd_mixed(x, r, w, 1e-5)
    for g in torch.autograd.grad(y, (x, r, w), torch.ones_like(y), create_graph=True):
        with pytest.raises(RuntimeError, match="no autograd formula"):
            torch.autograd.grad(g, (x, r, w), torch.ones_like(g), allow_unused=True, retain_graph=True)


def test_an_op_without_a_formula_refuses_forward_mode_and_functional_transforms(ops):
    x, w = meta(4, 128), meta(8, 128)
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError, match="forward-mode"):
        ops.linear_rows(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)), [w])
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda z: ops.linear_rows(z, [w.detach()]).sum())(x.detach())


def test_integer_outputs_carry_no_gradient(ops):
    assert not ops.topk_sample(meta(4, 128), meta(4, 128, grad=False), 3).requires_grad


@pytest.mark.parametrize("dtype", [torch.float32, BF16])
def test_the_loss_head_is_differentiable_in_its_incoming_gradient(ops, dtype):
    h, w, lam = meta(8, 16, dtype=dtype), meta(24, 16, dtype=dtype), torch.zeros((), device="meta", requires_grad=True)
    labels = torch.zeros(8, dtype=torch.long, device="meta")
    loss = lam * ops.fused_linear_ce(h, w, labels, -100, 2 if dtype == torch.float32 else 0, True)[0]
    for g in torch.autograd.grad(loss, (h, w), create_graph=True):
        (dlam,) = torch.autograd.grad(g.float().square().sum(), (lam,), retain_graph=True)
        assert dlam.shape == ()


def test_the_loss_head_passes_a_forward_mode_tangent_of_its_incoming_gradient(ops):
    h, w = meta(8, 16), meta(24, 16)
    loss = ops.fused_linear_ce(h, w, torch.zeros(8, dtype=torch.long, device="meta"), -100, 2, True)[0]
    fw = torch.autograd.forward_ad
    with fw.dual_level():
        up = fw.make_dual(torch.ones((), device="meta"), torch.ones((), device="meta"))
        for g in torch.autograd.grad(loss, (h, w), up):
            assert fw.unpack_dual(g).tangent is not None


def append_args(name, grad, base=None):
    caches = list(base) if base is not None else [heads(2).detach(), heads(2).detach()]
    new = [x if grad else x.detach() for x in (heads(4, 1), heads(2, 1), heads(2, 1))]
    return (*new, *tables(), 3, None, *((4, None) if name == "gqa_attn_decode_append" else ()), *caches,
            *((0.2,) if name == "gqa_attn_decode_append" else ())), caches


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("name", ["decode_rope_append", "gqa_attn_decode_append"])
def test_an_append_counts_as_a_write_to_the_caches(ops, name, grad):
    args, caches = append_args(name, grad)
    out = getattr(ops, name)(*args)
    assert [c._version for c in caches] == [1, 1] and out._version == 0
    assert not any(c.requires_grad for c in caches)
    both = meta(2, 2, 2, 8, 32, dtype=BF16, grad=False)  # the layers' caches as views of one tensor
    getattr(ops, name)(*append_args(name, grad, (both[0], both[1]))[0])
    assert both._version == 2
    with torch.inference_mode():  # inference tensors have no versions
        inference = [c.clone() for c in caches]
        getattr(ops, name)(*append_args(name, False, inference)[0])
    getattr(ops, name)(*append_args(name, False, inference)[0])


@pytest.mark.parametrize("name", ["decode_rope_append", "gqa_attn_decode_append"])
def test_a_cache_saved_for_backward_and_then_written_is_noticed(ops, name):
    args, (k_cache, _v_cache) = append_args(name, False)
    y = (k_cache * heads(2)).sum()
    getattr(ops, name)(*args)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


@pytest.mark.parametrize("name", ["gqa_rope_attn_fwd", "gqa_rope_attn_packed_fwd", "rope_fwd"])
def test_a_call_whose_tables_alone_require_a_gradient_is_recorded(ops, name):
    cos, sin = meta(8, 16), meta(8, 16, grad=False)
    q, k = heads(4).detach(), heads(2).detach()
    args = {"gqa_rope_attn_fwd": (q, k, k, cos, sin, 0.2), "rope_fwd": (q, k, cos, sin, False),
            "gqa_rope_attn_packed_fwd": (meta(2, 8, 8 * 32, dtype=BF16, grad=False), cos, sin, 4, 2, 0.2)}[name]
    out = getattr(ops, name)(*args)[0]
    assert out.requires_grad
    assert torch.autograd.grad(out, cos, torch.ones_like(out), allow_unused=True) == (None,)


def test_the_ops_have_their_autograd_from_the_import_on():
    """As an exported program calls them: no function of the package first."""
    code = """
import importlib, torch
importlib.import_module("mega-trading_amd")
x, w = (torch.empty(s, device="meta", requires_grad=True) for s in ((4, 16), (16,)))
y, _rstd = torch.ops.mega_trading_amd.rms_norm_fwd(x, w, 1e-5)
dx, dw = torch.autograd.grad(y, (x, w), torch.ones_like(y))
assert dx.shape == x.shape and dw.shape == w.shape
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    proc = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr[-2000:]
