"""The native dispatcher kernels (csrc/torch_binding.cpp) against the Python implementations they stand in for: the same bits
from both, for calls in canonical form and for calls that the native side hands over (views, index types that differ)."""

import pytest
import torch

import ops_rec
from helpers import small_case
from ops_rec import _activation, _dispatch, _ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def python_only():
    """Switches the native side off for one call, as replacing an allocator of ``_ops`` does."""

    def call(fn, *args):
        _dispatch.binding.set_native(False)
        try:
            return fn(*args)
        finally:
            _dispatch.binding.set_native(True)

    return call


def same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        assert x is None or (x.dtype == y.dtype and torch.equal(x, y))


@pytest.mark.parametrize("kw", [dict(), dict(delta=True), dict(rab=True, ctx=3, max_target=5, group=2), dict(heads=4, heads_k=2)],
                         ids=["equal", "delta", "bias", "grouped"])  # fmt: skip
@pytest.mark.parametrize("form", ["canonical", "view", "int64 targets"])
def test_attention_forward_and_gradients(kw, form, python_only):
    w = small_case(seed=9, batch=3, dim=64, lo=1, hi=150, dtype=torch.bfloat16, std=0.5, **kw).to(DEV)
    args = list(w.op_args())
    leaves = [t.clone().requires_grad_() for t in (w.q, w.k, w.v)] + ([w.attn_bias.clone().requires_grad_()] if w.attn_bias is not None else [])
    args[:3] = leaves[:3]
    if len(leaves) == 4:
        args[4] = leaves[3]
    if form == "view":
        args[0] = leaves[0].transpose(0, 1).contiguous().transpose(0, 1)
    if form == "int64 targets":
        args[-3] = torch.zeros(3, dtype=torch.int64, device=DEV) if args[-3] is None else args[-3].long()
        args[-4] = torch.zeros(3, dtype=torch.int64, device=DEV) if args[-4] is None else args[-4].long()

    def step():
        out = ops_rec.ascendc.attention.hstu_jagged(*args)
        return (out, *torch.autograd.grad(out.float().square().sum(), leaves))

    same(step(), python_only(step))


def test_a_replaced_allocator_sends_calls_through_python(monkeypatch):
    w = small_case(seed=2, batch=2, dim=64, lo=20, hi=90, dtype=torch.float16).to(DEV)
    made, plain = [], _ops._new_grad
    monkeypatch.setattr(_ops, "_new_grad", lambda like: (made.append(like.shape), plain(like))[1])
    grad = torch.randn_like(w.q)
    op = torch.ops.ops_rec.hstu_jagged_backward.equal
    op(grad, w.q, w.k, w.v, None, None, 0, w.max_seq_len, w.silu_scale, w.seq_offset)
    assert len(made) == 3
    monkeypatch.undo()
    op(grad, w.q, w.k, w.v, None, None, 0, w.max_seq_len, w.silu_scale, w.seq_offset)
    assert len(made) == 3


@pytest.mark.parametrize("m,split,with_bias", [(1, [16] * 4, True), (130, [64, 192, 128, 128], True), (77, [128] * 4, False)])
def test_projection_and_gradients_with_outputs_left_out(m, split, with_bias, python_only):
    n = sum(split)
    x, w, b = (torch.randn(s, device=DEV).to(d).requires_grad_() for s, d in (((m, 16), torch.bfloat16), ((n, 16), torch.bfloat16), ((n,), torch.float32)))
    bias = b if with_bias else None

    def step():
        u, v, q, k, lin = torch.ops.ops_rec.distance_in_linear_silu(x, w, bias, split)
        leaves = (x, w, b) if with_bias else (x, w)
        return (u, v, q, k, lin, *torch.autograd.grad((u.float().sum() + k.float().square().sum()), leaves))  # no gradient of v, q, lin

    same(step(), python_only(step))


def test_ln_mul(python_only):
    x, u = torch.randn(33, 96, device=DEV).half(), torch.randn(33, 96, device=DEV).half()
    g, b = torch.randn(96, device=DEV), torch.randn(96, device=DEV)
    step = lambda: (torch.ops.ops_rec.ln_mul(x, u, g, b), torch.ops.ops_rec.ln_mul(x.t().contiguous().t(), u, g, b))  # noqa: E731
    same(step(), python_only(step))
    same(step()[:1], (_activation.ln_mul(x, u, g, b),))


def test_memory_that_nobody_writes_is_filled_when_the_program_asks_for_it():
    """``torch.use_deterministic_algorithms`` has torch hand out new tensors full of NaN; what the native side allocates is no
    exception.  (Rows ahead of a non-zero first offset belong to no work item.)"""
    w = small_case(seed=4, batch=2, dim=64, lo=20, hi=60, dtype=torch.bfloat16).to(DEV)
    q, k, v = (torch.cat([torch.ones_like(t[:3]), t]) for t in (w.q, w.k, w.v))
    offs = w.seq_offset + 3
    call = lambda: torch.ops.ops_rec.hstu_jagged.equal(q, k, v, None, None, 0, w.max_seq_len, 0.0, offs)  # noqa: E731
    want = call()
    torch.zeros_like(want)  # (what the allocator hands out next holds zeros)
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        out = call()
    finally:
        torch.use_deterministic_algorithms(False)
    assert out[:3].isnan().all() and torch.equal(out[3:], want[3:])
