"""Which short lists of few items are cut into parts and which run without a list: both sides of each line of the rule, each result against
the CPU oracle and against the other route (HSTU_MI355_SPLIT=1 cuts wherever the list is short enough).

The routes add the same products in fp32, in another order: 16-bit outputs are at most one rounding step apart, 2^-7 of the value in bf16
and 2^-10 in fp16, and 2e-7 where a value is next to zero.
"""

import pytest
import torch

import helpers
import ops_rec  # noqa: F401
from ops_rec import _ops, workloads
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, FP = torch.bfloat16, torch.float16


def prepared(w):
    k_offs = w.seq_offset if w.seq_offset_k is None else w.seq_offset_k
    max_k = w.max_seq_len if w.max_seq_len_k is None else w.max_seq_len_k
    return _ops.prepare_forward(w.q, w.k, w.v, None, w.attn_bias, 0, w.max_seq_len, max_k, w.silu_scale, w.seq_offset, k_offs,
                                w.num_context, w.num_target, w.target_group_size, w.alpha)  # fmt: skip


@pytest.mark.parametrize(
    "lengths,heads,dim,dtype,history,kw,cut",
    [
        ([1000, 900] * 4, 1, 64, BF, 0, dict(), False),  # 64 slots of at most 1024 keys
        ([1000, 900] * 3 + [1000], 1, 64, BF, 0, dict(), True),  # 56 slots
        ([1024] * 8, 1, 64, FP, 0, dict(), False),
        ([1025] * 8, 1, 64, FP, 0, dict(), True),  # causal rows longer than that
        ([200, 130] * 8, 2, 64, FP, 1300, dict(), False),  # rows on a history, up to 2048 keys
        ([200, 130] * 8, 2, 128, BF, 1848, dict(), False),
        ([200, 130] * 8, 2, 128, BF, 1849, dict(), True),  # past 2048 keys
        ([700, 650] * 6, 1, 64, BF, 0, dict(num_context=3, max_target=9), True),  # context rows
        ([700, 650] * 6, 1, 64, BF, 0, dict(rab_std=0.2), True),  # 72 slots with a bias
        ([700, 650] * 11, 1, 64, BF, 0, dict(rab_std=0.2), False),  # 132
        ([600] * 20, 2, 64, FP, 0, dict(max_target=30, target_group_size=3, heads_k=1), False),
    ],
    ids=str,
)
def test_both_sides_of_the_rule(lengths, heads, dim, dtype, history, kw, cut, monkeypatch):
    w = workloads.make("rule", batch=len(lengths), heads=heads, dim=dim, lo=0, hi=0, lengths=lengths, dtype=dtype, std=0.5,
                       seed=len(lengths) + dim, **kw)  # fmt: skip
    if history:
        lk = [n + history for n in lengths]
        gen = torch.Generator().manual_seed(1)
        w.seq_offset_k = torch.tensor([0] + lk).cumsum(0).to(w.seq_offset.dtype)
        w.max_seq_len_k = max(lk)
        w.k, w.v = ((torch.randn(sum(lk), t.shape[1], t.shape[2], generator=gen) * 0.5).to(dtype) for t in (w.k, w.v))
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")  # (slot 128 has a kernel of its own for some of these)
    d = w.to(DEV)
    p = prepared(d)
    assert p.kernel_name().endswith("_split") == cut, p.kernel_name()
    assert (p.workspace_bytes > 0) == cut
    out = p.launch().clone()
    ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "1")
    other = prepared(d)
    assert other.kernel_name().endswith("_split"), other.kernel_name()
    torch.testing.assert_close(out.float(), other.launch().float(), atol=2e-7, rtol=2**-7 if dtype == BF else 2**-10)
