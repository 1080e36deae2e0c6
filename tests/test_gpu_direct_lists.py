"""Plain launches without a work list (a workgroup per (level, pair, head) slot, chosen while every slot is resident or sweeps are
short) against the CPU oracle: pair counts that are not a multiple of 8, grouped heads, empty sequences, context rows (whose
first tile heads the list), rows past the last offset, and, with more slots than resident workgroups, both sides of the rule's
bound on the keys."""

import pytest
import torch

import helpers
import ops_rec
from oracle import hstu_oracle as O
from ops_rec import _ops, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dim,dtype", [(32, torch.float16), (64, torch.bfloat16), (128, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("lengths,kw,list_free", [
    ([1], dict(), True), ([300, 0, 129, 128, 1], dict(), True), ([130, 64, 257], dict(heads_k=1, rab_std=0.3), True),
    ([200, 90, 384, 33, 2, 7, 256], dict(num_context=3, max_target=9, target_group_size=2), True), ([90] * 700, dict(), "up to slot 128"),
    ([385] * 3, dict(rab_std=0.2), True), ([384] + [40] * 199, dict(), "up to slot 128"), ([385] + [40] * 199, dict(), False),
], ids=["one row", "ragged", "grouped bias", "context", "many", "long but few", "at the bound", "past the bound"])  # fmt: skip
def test_against_the_oracle(lengths, kw, list_free, dim, dtype, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")  # (the kernels for short and tiny lists would take some of these)
    if len(lengths) > 200:
        lengths = lengths[: 700 if dim <= 64 else 350]
    w = workloads.make("direct", batch=len(lengths), heads=2, dim=dim, lo=0, hi=0, lengths=lengths, dtype=dtype, std=0.5,
                       seed=dim + len(lengths), **kw)  # fmt: skip
    wd = w.to(DEV)
    extra = torch.randn(5, 2, dim, device=DEV).to(dtype)  # rows past the last offset
    wd.q = torch.cat([wd.q, extra])
    p = _ops.prepare_forward(wd.q, wd.k, wd.v, None, wd.attn_bias, 0, wd.max_seq_len, wd.max_seq_len, wd.silu_scale, wd.seq_offset,
                             wd.seq_offset, wd.num_context, wd.num_target, wd.target_group_size, wd.alpha)  # fmt: skip
    assert p.kernel_name().endswith("_direct") == (dim <= 128 if list_free == "up to slot 128" else list_free), p.kernel_name()
    out = ops_rec.ascendc.attention.hstu_jagged(*wd.op_args())
    assert not out[-5:].any()
    ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
    torch.testing.assert_close(out[:-5].float().cpu(), ref, atol=1e-2, rtol=1e-2)
