"""attn_bias values that no visible (row, key) pair reads -- rows behind a sequence, keys behind it, keys the causal mask hides --
may be anything: outputs and gradients are the same bits with NaN or infinities there, at row lengths where a 32-key block ends
inside, at and behind a row."""

import itertools

import pytest
import torch

import helpers
import ops_rec  # noqa: F401
from oracle import hstu_oracle as oracle

pytestmark = pytest.mark.gpu


def planes(max_len, lengths, heads, where, dtype=torch.bfloat16):
    """The same attn_bias twice, the second with what no pair reads replaced."""
    gen = torch.Generator(device="cuda").manual_seed(1)
    clean = (torch.randn(len(lengths), heads, max_len, max_len, generator=gen, device="cuda") * 0.3).to(dtype)
    dirty = clean.clone()
    if where == "hidden":
        above = torch.ones(max_len, max_len, dtype=torch.bool, device="cuda").triu(1)
        dirty[:, :, above] = float("-inf")
    for b, n in enumerate(lengths):
        if where == "rows":
            dirty[b, :, n:, :] = float("nan")
        elif where == "keys":
            dirty[b, :, :n, n:] = float("nan")
    return clean, dirty


@pytest.mark.parametrize("where", ["rows", "keys", "hidden"])
@pytest.mark.parametrize("max_len", [298, 300, 301, 304, 320])
@pytest.mark.parametrize(
    "dim,order,dtype",
    [(dim, order, torch.bfloat16) for dim in (64, 128, 256) for order in ("0", "1", "2", "3")]
    + [(320, None, torch.bfloat16), (60, None, torch.float16), (64, None, torch.float32)],
    ids=str,
)
def test_bias_that_no_pair_reads_reaches_no_gradient(dim, order, dtype, max_len, where, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", order)
    lengths, heads = [max_len - 7, max_len - 40, max_len, 97], 2
    gen = torch.Generator(device="cuda").manual_seed(0)

    def rand(*shape):
        return (torch.randn(*shape, generator=gen, device="cuda") * 0.3).to(dtype)

    rows = sum(lengths)
    q, k = (rand(rows, heads, dim) for _ in range(2))
    v, grad = (rand(rows, heads, dim // 16 * 16) for _ in range(2))
    offsets = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32, device="cuda")
    clean, dirty = planes(max_len, lengths, heads, where, dtype)

    def run(bias):
        return torch.ops.ops_rec.hstu_jagged_backward.equal(
            grad, q, k, v, None, bias, 0, max_len, 1.0 / max_len, offsets, None, None, 0, dim**-0.5
        )[:4]

    for want, got in zip(run(clean), run(dirty)):
        assert torch.equal(want, got)


@pytest.mark.parametrize("where", ["rows", "keys"])
@pytest.mark.parametrize("max_len", [298, 300, 301, 304])
@pytest.mark.parametrize("biased", [False, True])
def test_mask_values_past_a_sequence_reach_nothing(biased, max_len, where):
    lengths, heads, dim = [max_len - 7, max_len - 40, max_len, 97], 2, 64
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v, grad = ((torch.randn(sum(lengths), heads, dim, generator=gen, device="cuda") * 0.3).bfloat16() for _ in range(4))
    offsets = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32, device="cuda")
    bias = planes(max_len, lengths, heads, "rows")[0] if biased else None
    results = []
    for mask in planes(max_len, lengths, heads, where):
        rest = (mask, bias, 3, max_len, 1.0 / max_len, offsets, None, None, 0, dim**-0.5)
        out = torch.ops.ops_rec.hstu_jagged.equal(q, k, v, *rest)
        results.append((out, *torch.ops.ops_rec.hstu_jagged_backward.equal(grad, q, k, v, *rest)[: 4 if biased else 3]))
    for want, got in zip(*results):
        assert torch.equal(want, got)


@pytest.mark.parametrize("where", ["rows", "keys", "hidden"])
@pytest.mark.parametrize("max_len", [298, 301, 304, 1310, 1311, 1312])
@pytest.mark.parametrize(
    "dim,dtype,heads,switches",
    [
        (32, torch.bfloat16, 2, {}),
        (64, torch.float16, 2, {}),
        (64, torch.bfloat16, 2, {"SPLIT": "1", "SHORT": "0"}),  # (long items in parts)
        (128, torch.bfloat16, 2, {}),
        (128, torch.bfloat16, 2, {"SHORT": "0"}),
        (128, torch.float16, 16, {"SHORT": "0", "SPLIT": "0"}),  # (from a list)
        (256, torch.bfloat16, 2, {}),
        (320, torch.bfloat16, 2, {}),
        (60, torch.bfloat16, 2, {}),
        (64, torch.float32, 2, {}),
    ],
    ids=str,
)
def test_bias_that_no_pair_reads_reaches_no_output(dim, dtype, heads, switches, max_len, where, monkeypatch):
    for name, value in switches.items():
        helpers.set_switch(monkeypatch, f"HSTU_MI355_{name}", value)
    lengths = [max_len - 7, max_len - 40, max_len, 97]
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = ((torch.randn(sum(lengths), heads, dim // 16 * 16 if i == 2 else dim, generator=gen, device="cuda") * 0.3).to(dtype) for i in range(3))
    offsets = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32, device="cuda")
    want, got = (
        torch.ops.ops_rec.hstu_jagged.equal(q, k, v, None, bias, 0, max_len, 1.0 / max_len, offsets, None, None, 0, dim**-0.5)
        for bias in planes(max_len, lengths, heads, where, dtype)
    )
    assert torch.equal(want, got)


@pytest.mark.parametrize("max_len", [301, 304, 1312])
@pytest.mark.parametrize("dim", [64, 128, 256])
def test_hidden_bias_under_context_rows_and_target_groups(dim, max_len, monkeypatch):
    """What the mask hides with context rows in front and target rows behind, by the mask itself."""
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    lengths, heads, context, targets, group = [max_len - 7, max_len - 40, max_len, 197], 2, 37, 70, 3
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = ((torch.randn(sum(lengths), heads, dim, generator=gen, device="cuda") * 0.3).bfloat16() for _ in range(3))
    count = lambda n: torch.full((len(lengths),), n, dtype=torch.int32, device="cuda")  # noqa: E731
    offsets = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32, device="cuda")
    clean, _ = planes(max_len, lengths, heads, "rows")
    dirty = torch.full_like(clean, float("nan"))
    for b, n in enumerate(lengths):
        seen = torch.from_numpy(oracle.builtin_mask(n, n, context, targets, group)).cuda() != 0
        dirty[b, :, :n, :n] = torch.where(seen, clean[b, :, :n, :n], torch.tensor(float("nan"), dtype=clean.dtype, device="cuda"))
    want, got = (
        torch.ops.ops_rec.hstu_jagged.equal(q, k, v, None, bias, 0, max_len, 1.0 / max_len, offsets, count(context), count(targets), group, dim**-0.5)
        for bias in (clean, dirty)
    )
    assert torch.equal(want, got)
