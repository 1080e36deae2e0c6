"""The native dispatcher kernels (csrc/torch_binding.cpp) against the Python implementations they stand in for: the same bits
from both, for calls in canonical form and for calls that the native side hands over (views, index types that differ)."""

import dataclasses

import pytest
import torch

import ops_rec
import helpers
from helpers import small_case
from ops_rec import _activation, _dispatch, _ops, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        assert x is None or (x.dtype == y.dtype and torch.equal(x, y))


@pytest.mark.parametrize("kw", [dict(), dict(delta=True), dict(rab=True, ctx=3, max_target=5, group=2), dict(heads=4, heads_k=2)],
                         ids=["equal", "delta", "bias", "grouped"])  # fmt: skip
@pytest.mark.parametrize("form", ["canonical", "view", "int64 targets"])
def test_attention_forward_and_gradients(kw, form):
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

    out = ops_rec.ascendc.attention.hstu_jagged(*args)
    grad = torch.randn_like(out)
    got = (out, *torch.autograd.grad(out, leaves, grad))
    # the same through the Python implementations
    with torch.no_grad():
        want = (_ops.hstu_jagged_delta if w.seq_offset_k is not None else _ops.hstu_jagged_equal)(*args)
        d = dataclasses.replace(w, q=args[0], num_target=args[-3], num_context=args[-4])
        grads = _ops.hstu_jagged_backward_delta(*helpers.backward_args(d, grad))
    same(got, (want, *grads[: len(leaves)]))


@pytest.mark.parametrize("m,split,with_bias", [(1, [16] * 4, True), (130, [64, 192, 128, 128], True), (77, [128] * 4, False)])
def test_projection_and_gradients_with_outputs_left_out(m, split, with_bias):
    n = sum(split)
    x, w, b = (torch.randn(s, device=DEV).to(d).requires_grad_() for s, d in (((m, 16), torch.bfloat16), ((n, 16), torch.bfloat16), ((n,), torch.float32)))
    bias = b if with_bias else None
    leaves = (x, w, b) if with_bias else (x, w)
    outs = torch.ops.ops_rec.distance_in_linear_silu(x, w, bias, split)
    gu, gk = torch.randn_like(outs[0]), torch.randn_like(outs[3])
    got = (*outs, *torch.autograd.grad((outs[0], outs[3]), leaves, (gu, gk)))  # no gradient of v, q, lin
    with torch.no_grad():
        want = _activation.distance_in_linear_silu(x, w, bias, split)
        grads = _activation.in_linear_silu_backward(x, w, bias, gu, torch.zeros_like(outs[1]), torch.zeros_like(outs[2]), gk, want[4], split)
    same(got, (*want, *grads[: len(leaves)]))


def test_ln_mul():
    x, u = torch.randn(33, 96, device=DEV).half(), torch.randn(33, 96, device=DEV).half()
    g, b = torch.randn(96, device=DEV), torch.randn(96, device=DEV)
    view = x.t().contiguous().t()
    op = torch.ops.ops_rec.ln_mul
    same((op(x, u, g, b), op(view, u, g, b)), (_activation.ln_mul(x, u, g, b), _activation.ln_mul(view, u, g, b)))


def test_memory_that_nobody_writes_is_filled_when_the_program_asks_for_it(monkeypatch):
    """``torch.use_deterministic_algorithms`` has torch hand out new tensors full of NaN; what the native side allocates is no
    exception.  (Rows ahead of a non-zero first offset belong to no work item.)"""
    w = small_case(seed=4, batch=2, dim=64, lo=20, hi=60, dtype=torch.bfloat16).to(DEV)
    q, k, v = (torch.cat([torch.ones_like(t[:3]), t]) for t in (w.q, w.k, w.v))
    offs = w.seq_offset + 3
    call = lambda: torch.ops.ops_rec.hstu_jagged.equal(q, k, v, None, None, 0, w.max_seq_len, 0.0, offs)  # noqa: E731
    want = call()
    torch.zeros_like(want)  # (what the allocator hands out next holds zeros)
    helpers.poison_workspace(monkeypatch)
    out = call()
    assert out[:3].isnan().all() and torch.equal(out[3:], want[3:])


@pytest.mark.parametrize("delta", [False, True], ids=["equal", "delta"])
def test_offsets_that_serve_both_sides_are_saved_once(delta, monkeypatch):
    """Hooks that copy what is saved leave the backward with the workspace of self-attention (offsets that are one tensor)."""
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "2")
    w = workloads.make("saved", dtype=torch.bfloat16, device=DEV, seed=5, batch=4, heads=2, dim=64, lo=500, hi=512, max_seq_len=512)
    leaves = [t.requires_grad_() for t in (w.q, w.k, w.v)]
    grad = torch.randn_like(w.q)
    packed = []

    def workspace(pack):
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            if delta:
                out = torch.ops.ops_rec.hstu_jagged.delta(*leaves, None, None, 0, 512, 512, 1.0, w.seq_offset, w.seq_offset, None, None, 0, w.alpha)
            else:
                out = torch.ops.ops_rec.hstu_jagged.equal(*leaves, None, None, 0, 512, 1.0, w.seq_offset, None, None, 0, w.alpha)
        return helpers.allocated_beside(lambda: torch.autograd.grad(out, leaves, grad, retain_graph=True))

    want, size = workspace(lambda t: t)
    got, copied = workspace(lambda t: (packed.append(t), t.clone())[1])
    assert len(packed) == 4 and copied == size > 0
    same(got, want)


def test_a_backward_whose_workspace_does_not_fit(monkeypatch):
    """The native kernel's answer to an allocator that has no room for the workspace is the launch order that needs none."""
    w = workloads.make("oom", dtype=torch.bfloat16, device=DEV, seed=3, batch=8, heads=4, dim=128, lo=1500, hi=2048, max_seq_len=2048)
    args = helpers.backward_args(w, torch.randn_like(w.q))
    call = lambda: ops_rec.ascendc.attention.hstu_jagged_backward(*args)  # noqa: E731
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "0")
    want = call()
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "2")
    assert helpers.allocated_beside(call)[1] > 64 << 20
    got, refused = helpers.with_room_for(call, 32 << 20, like=want)
    assert refused == 1 and all((a is None and b is None) or torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("python", [False, True], ids=["native", "python"])
def test_a_backward_with_room_for_the_smaller_workspace(python, monkeypatch):
    """Context rows, whole layouts: the dS of the three-launch order needs a few MiB less than the tiles, and is what the call takes
    where those do not fit."""
    w = workloads.make("oom", dtype=torch.bfloat16, device=DEV, seed=3, batch=4, heads=8, dim=128, lo=0, hi=0,
                       lengths=[2052, 2052, 2016, 2006], max_seq_len=2052, num_context=4)  # fmt: skip
    args = helpers.backward_args(w, torch.randn_like(w.q))
    op = _ops.hstu_jagged_backward_delta if python else ops_rec.ascendc.attention.hstu_jagged_backward
    call = lambda: op(*args)  # noqa: E731
    tiles = helpers.allocated_beside(call)[1]
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "1")
    want, plane = helpers.allocated_beside(call)
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", None)
    assert plane + (4 << 20) <= tiles
    got, refused = helpers.with_room_for(call, (plane + (2 << 20)) // (2 << 20) * (2 << 20), like=want)
    assert refused == 1 and all((a is None and b is None) or torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("k", [1024, 1040])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_projection_backward_on_both_sides_of_the_rule_for_its_weight_gradient(k, dtype):
    m, split = 77, [k] * 4
    x, w, b = torch.randn(m, k, device=DEV).to(dtype), (torch.randn(4 * k, k, device=DEV) / 32).to(dtype), torch.randn(4 * k, device=DEV)
    lin = torch.ops.ops_rec.distance_in_linear_silu(x, w, b, split)[4]
    grads = [torch.randn(m, k, device=DEV).to(dtype) for _ in range(4)]
    call = lambda: torch.ops.ops_rec.in_linear_silu_backward(x, w, b, *grads, lin, split)  # noqa: E731
    (dx, dw, db, _), workspace = helpers.allocated_beside(call)
    assert (workspace >= 4 * dw.numel()) == (k <= 1024)  # fp32 partial outputs, or none
    same((dx, dw, db), _activation.in_linear_silu_backward(x, w, b, *grads, lin, split)[:3])
    d_mixed, own_dw, own_db = _activation.silu_backward_with_weight(lin, grads, split, x)
    for got, other in ((dw, own_dw), (dw, d_mixed.double().t() @ x.double()), (db, own_db)):
        assert (got.double() - other.double()).norm() <= 5e-3 * other.double().norm()


@pytest.mark.parametrize("python", [False, True], ids=["native", "python"])
def test_a_projection_backward_whose_workspace_does_not_fit(python):
    """Without room for the partial weight gradients the weight gradient is a product of what the element-wise stage left."""
    m, k, split = 3000, 1024, [1024] * 4
    x, w, b = torch.randn(m, k, device=DEV).bfloat16(), torch.randn(4096, k, device=DEV).bfloat16() / 32, torch.randn(4096, device=DEV)
    lin = torch.ops.ops_rec.distance_in_linear_silu(x, w, b, split)[4]
    grads = [torch.randn(m, 1024, device=DEV).bfloat16() for _ in range(4)]
    op = _activation.in_linear_silu_backward if python else torch.ops.ops_rec.in_linear_silu_backward
    call = lambda: op(x, w, b, *grads, lin, split)  # noqa: E731
    want, workspace = helpers.allocated_beside(call)
    assert _dispatch.binding is not None and workspace > 60 << 20
    got, refused = helpers.with_room_for(call, 40 << 20, like=(*want, lin))
    assert refused == 1
    for a, e in zip(got[:3], want[:3]):
        assert a.dtype == e.dtype and (a.double() - e.double()).norm() <= 5e-3 * e.double().norm()
