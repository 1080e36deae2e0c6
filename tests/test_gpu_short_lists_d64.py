"""The forward kernel for short work lists at the head-dim slots 64 and 32 (three workgroups of eight 16-row wavefronts per compute unit; four of
the wavefronts bring K and four V), forced with HSTU_MI355_SHORT=1, against the CPU oracle: tile and sub-tile edges, padded head dims, masks,
grouped heads, keys of their own, outputs on addresses that take no 16-byte stores, with and without attn_bias."""

import pytest
import torch

import ops_rec
from ops_rec import _ops, workloads
from oracle import hstu_oracle as O
import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def kernel_name(w):
    k_offs = w.seq_offset_k if w.seq_offset_k is not None else w.seq_offset
    p = _ops.prepare_forward(w.q, w.k, w.v, w.mask, w.attn_bias, w.mask_type, w.max_seq_len,
                             w.max_seq_len_k or w.max_seq_len, w.silu_scale, w.seq_offset, k_offs, w.num_context,
                             w.num_target, w.target_group_size, w.alpha)  # fmt: skip
    return p.kernel_name()


CASES = {
    "sub-tile edges": dict(heads=2, lengths=[31, 32, 33, 65, 1, 0, 96, 97]),
    "tile edges": dict(heads=1, lengths=[127, 128, 129, 255, 257, 1000, 1024]),
    "nine pairs": dict(heads=1, lengths=[140, 3, 139, 70, 128, 1, 100, 64, 90]),
    "context, targets, groups": dict(heads=2, lengths=[20, 400, 131, 260], num_context=5, max_target=17, target_group_size=3),
    "grouped heads": dict(heads=4, heads_k=2, lengths=[200, 129, 30, 1]),
    "padded head dims": dict(heads=2, dim=48, dim_v=48, lengths=[260, 100, 33]),
    "slot 32": dict(heads=4, heads_k=2, dim=32, lengths=[260, 100, 33, 128], num_context=3, max_target=9, target_group_size=2),
    "dims of 16": dict(heads=2, dim=16, lengths=[129, 300, 32, 1]),
    "64-key edges": dict(heads=2, lengths=[63, 64, 65, 191, 192, 193]),
    "narrow v": dict(heads=2, dim=64, dim_v=16, lengths=[260, 100, 33]),
    "odd pitch of the bias": dict(heads=2, lengths=[300, 150], max_seq_len=308),
    "int64 offsets": dict(heads=3, lengths=[100, 700, 350], index_dtype=torch.int64),
}


@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("name", list(CASES))
def test_against_the_oracle(name, dtype, bias, monkeypatch):
    kw = dict(dict(dim=64), **CASES[name])
    if bias:
        kw["rab_std"] = 0.5
        kw.setdefault("max_seq_len", -(-max(kw["lengths"]) // 4) * 4)
    w = workloads.make("short", batch=len(kw["lengths"]), lo=0, hi=0, dtype=dtype, std=0.5, seed=len(name), **kw)
    wd = w.to(DEV)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "1")
    assert kernel_name(wd).endswith("_d64_rab_short" if bias else "_d64_short"), kernel_name(wd)
    got = ops_rec.ascendc.attention.hstu_jagged(*wd.op_args()).float().cpu()
    ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
    torch.testing.assert_close(got, ref, atol=1e-2, rtol=1e-2)
    lo = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=dtype, emulate_lowp=dtype, **w.oracle_kwargs()).float()
    assert O.mismatch_fraction(got, lo, 5e-3) < 5e-3


@pytest.mark.parametrize("rows,keys", [(1, 33), (127, 1000), (128, 31), (129, 64), (501, 1000)])
def test_keys_of_their_own_and_rows_past_the_last(rows, keys, monkeypatch):
    torch.manual_seed(rows)
    batch, heads, dim = 3, 2, 64
    q = torch.randn(batch * rows + 5, heads, dim, dtype=torch.float16) * 0.5
    k, v = (torch.randn(batch * keys, heads, dim, dtype=torch.float16) * 0.5 for _ in range(2))
    offs, offs_k = (torch.arange(batch + 1, dtype=torch.int32) * n for n in (rows, keys))
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "1")
    q_len = max(rows, 65)  # (more than 64 rows by the bound: the kernels for few rows stay out)
    args = (None, None, 0, q_len, keys, 1.0 / keys, offs.to(DEV), offs_k.to(DEV), None, None, 0, dim**-0.5)
    p = _ops.prepare_forward(q.to(DEV), k.to(DEV), v.to(DEV), None, None, 0, q_len, keys, 1.0 / keys, args[6], args[7], None, None, 0, dim**-0.5)
    assert p.kernel_name() == "hstu_fwd_f16_d64_short", p.kernel_name()
    got = ops_rec.ascendc.attention.hstu_jagged(q.to(DEV), k.to(DEV), v.to(DEV), *args).float().cpu()
    assert not got[-5:].any()
    ref = torch.zeros(batch * rows, heads, dim, dtype=torch.float64)
    for b in range(batch):
        qs, ks, vs = q[b * rows : (b + 1) * rows].double(), k[b * keys : (b + 1) * keys].double(), v[b * keys : (b + 1) * keys].double()
        for h in range(heads):
            s = qs[:, h] @ ks[:, h].T * dim**-0.5
            seen = torch.arange(keys)[None, :] <= torch.arange(rows)[:, None] + (keys - rows)
            ref[b * rows : (b + 1) * rows, h] = (torch.nn.functional.silu(s) / keys * seen) @ vs[:, h]
    torch.testing.assert_close(got[:-5].double(), ref, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("batch,rows,keys,bias,short,dim", [(*c, 64) for c in (
    (32, 1024, 1024, False, True), (32, 1024, 1025, False, False), (3, 300, 704, False, True), (3, 300, 708, False, False),
    (64, 300, 708, False, True), (256, 1024, 1024, False, True), (257, 1024, 1024, False, False), (2, 66, 66, False, True),
    (4, 512, 512, True, True), (4, 516, 516, True, False), (64, 256, 256, True, True), (64, 260, 260, True, False),
)] + [(*c, 32) for c in (
    (16, 500, 704, False, True), (16, 500, 705, False, False), (64, 500, 500, False, False), (80, 500, 512, False, True), (80, 500, 513, False, False),
    (64, 256, 256, True, True), (65, 256, 256, True, False), (16, 512, 512, True, True), (17, 512, 512, True, False), (16, 516, 516, True, False),
)], ids=str)  # fmt: skip
def test_the_rule(batch, rows, keys, bias, short, dim):
    """Which calls of 4 heads take the kernel by themselves: bounds on keys, K / V bytes, slots; 256 compute units."""
    q = torch.empty(batch * rows, 4, dim, dtype=torch.bfloat16, device=DEV)
    k = torch.empty(batch * keys, 4, dim, dtype=torch.bfloat16, device=DEV)
    offs, offs_k = ((torch.arange(batch + 1, dtype=torch.int32) * n).to(DEV) for n in (rows, keys))
    rab = torch.empty(batch, 4, rows, keys, dtype=torch.bfloat16, device=DEV) if bias else None
    p = _ops.prepare_forward(q, k, k, None, rab, 0, rows, keys, 1.0 / keys, offs, offs_k, None, None, 0, 0.125)
    assert p.kernel_name().endswith("_short") == short, p.kernel_name()
