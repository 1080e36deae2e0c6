"""attn_bias values that no visible (row, key) pair reads -- rows behind a sequence, keys behind it, keys the causal mask hides --
may be anything: the gradients are the same bits with NaN or infinities there, at row lengths where a 32-key block ends inside,
at and behind a row."""

import itertools

import pytest
import torch

import ops_rec  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["rows", "keys", "hidden"])
@pytest.mark.parametrize("max_len", [298, 300, 301, 304, 320])
@pytest.mark.parametrize("dim", [64, 128, 256])
def test_bias_that_no_pair_reads_reaches_no_gradient(dim, max_len, where):
    lengths, heads = [max_len - 7, max_len - 40, max_len, 97], 2
    gen = torch.Generator(device="cuda").manual_seed(0)

    def rand(*shape):
        return (torch.randn(*shape, generator=gen, device="cuda") * 0.3).bfloat16()

    rows = sum(lengths)
    q, k, v, grad = (rand(rows, heads, dim) for _ in range(4))
    offsets = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32, device="cuda")
    clean = rand(len(lengths), heads, max_len, max_len)
    dirty = clean.clone()
    if where == "hidden":
        above = torch.ones(max_len, max_len, dtype=torch.bool, device="cuda").triu(1)
        dirty[:, :, above] = float("-inf")
    for b, n in enumerate(lengths):
        if where == "rows":
            dirty[b, :, n:, :] = float("nan")
        elif where == "keys":
            dirty[b, :, :n, n:] = float("nan")

    def run(bias):
        return torch.ops.ops_rec.hstu_jagged_backward.equal(
            grad, q, k, v, None, bias, 0, max_len, 1.0 / max_len, offsets, None, None, 0, dim**-0.5
        )[:4]

    for want, got in zip(run(clean), run(dirty)):
        assert torch.equal(want, got)
