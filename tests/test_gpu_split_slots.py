"""Rows on a history in launches without a list whose items are all cut alike, paged and not: edges of tiles, parts and pages against the CPU
oracle and against whole items (HSTU_MI355_SPLIT=0).

Parts add the same products in fp32, in another order: 16-bit outputs are at most one rounding step apart, 2^-7 of the value in bf16 and 2^-10 in
fp16, and 2e-7 where a value is next to zero.
"""

import pytest
import torch

import helpers
import ops_rec
from ops_rec import _ops, workloads
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, FP = torch.bfloat16, torch.float16


def offsets(lengths):
    return torch.tensor([0] + lengths).cumsum(0)


CASES = {  # rows and keys of each sequence
    "one tile": (dict(heads=3, dim=128), [1, 31, 32, 33, 96, 127, 128], [3000, 2600, 2049, 2080, 2111, 2500, 2700], BF),
    "parts without keys": (dict(heads=2, dim=128), [128, 5, 0, 64], [4000, 5, 0, 100], FP),
    "fewer keys than rows": (dict(heads=1, dim=64), [100, 128, 70], [30, 2500, 0], BF),
    "two tiles": (dict(heads=4, heads_k=2, dim=64), [129, 256, 200, 130, 1], [2100, 3000, 2600, 2300, 2200], FP),
    "four tiles, targets": (dict(heads=2, dim=96, max_target=40, target_group_size=3), [400, 512, 130], [2500, 2700, 3000], BF),
    "slot 256": (dict(heads=2, dim=256), [1, 128, 77], [2500, 4000, 2049], FP),
    "slot 256, odd dims": (dict(heads=4, heads_k=1, dim=200, dim_v=144), [200, 129, 256], [2500, 2100, 2300], BF),
    "64-bit offsets": (dict(heads=2, dim=128, index_dtype=torch.int64), [64, 100, 12], [2500, 2100, 2300], BF),
    "one pair": (dict(heads=1, dim=128), [200], [4000], BF),
    "slots not in eights": (dict(heads=5, dim=128), [128, 100, 1, 128, 127], [5000, 3000, 2049, 100, 4100], FP),
    "no mask": (dict(heads=2, dim=64), [64, 100, 12], [2500, 2100, 2300], BF),
}


@pytest.mark.parametrize("name", list(CASES))
def test_rows_on_a_history(name, monkeypatch):
    kw, rows, keys, dtype = CASES[name]
    w = workloads.make(name, batch=len(rows), lo=0, hi=0, lengths=rows, dtype=dtype, std=0.5, seed=len(name), **kw)
    if kw.get("max_target"):  # (targets come on top of the rows)
        rows = (w.seq_offset[1:] - w.seq_offset[:-1]).tolist()
        keys = [a + b for a, b in zip(rows, keys)]
    w.mask_type = 2 if name == "no mask" else 0
    gen = torch.Generator().manual_seed(1)
    w.seq_offset_k, w.max_seq_len_k = offsets(keys).to(w.seq_offset.dtype), max(keys)
    w.k, w.v = ((torch.randn(sum(keys), t.shape[1], t.shape[2], generator=gen) * 0.5).to(dtype) for t in (w.k, w.v))
    d = w.to(DEV)

    def prepared():
        return _ops.prepare_forward(d.q, d.k, d.v, None, None, d.mask_type, d.max_seq_len, d.max_seq_len_k, d.silu_scale, d.seq_offset,
                                    d.seq_offset_k, d.num_context, d.num_target, d.target_group_size, d.alpha)  # fmt: skip

    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "1")
    p = prepared()
    assert p.kernel_name().endswith("_split") and p.workspace_bytes > 0, p.kernel_name()
    out = p.launch().clone()
    for _ in range(2):  # (the arrival counters are back at zero)
        assert torch.equal(p.launch(), out)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    whole = prepared()
    assert not whole.kernel_name().endswith("_split")
    torch.testing.assert_close(out.float(), whole.launch().float(), atol=2e-7, rtol=2**-7 if dtype == BF else 2**-10)
    ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)


NAMES = ("seq_offset", "seq_offset_k", "page_offsets", "page_ids", "last_page_len", "num_target")


@pytest.mark.parametrize(
    "hist,prev,targets,kw",
    [
        ([60, 1, 32, 90], [2000, 700, 1300, 64], [32, 1, 31, 6], dict(heads=3, dim=128, page_size=128)),  # new rows start inside a sub-tile
        ([64, 96, 32], [1024, 960, 992], [1, 32, 64], dict(heads=4, heads_k=2, dim=64, page_size=32, dtype=FP)),  # and on an edge
        ([10, 3], [3000, 0], [50, 4], dict(heads=2, dim=256, page_size=64)),  # parts without keys
        ([200, 130, 300], [2000, 1500, 1800], [20, 60, 7], dict(heads=2, dim=192, page_size=256, dtype=FP)),  # three tiles
        ([20] * 70, [300] * 70, [9] * 70, dict(heads=4, dim=128, page_size=64)),  # whole items, a workgroup each
        ([33, 64], [1500, 2500], [10, 20], dict(heads=2, dim=128, page_size=128, index_dtype=torch.int64)),
    ],
    ids=str,
)
def test_paged(hist, prev, targets, kw, monkeypatch):
    kw = dict(dict(dtype=BF), **kw)
    c = helpers.paged_case(hist=hist, prev=prev, targets=targets, std=0.3, seed=len(hist), **kw)
    alpha = kw["dim"] ** -0.5
    d = {n: (t.to(DEV) if torch.is_tensor(t) else t) for n, t in c.items()}

    def run():
        return ops_rec.ascendc.attention.hstu_paged(
            d["q"], d["k"], d["v"], d["kv_cache"], mask_type=0, max_seq_len=c["max_seq_len"], max_seq_len_k=c["max_seq_len_k"],
            seq_offset_t=d["seq_offset_t"], target_group_size=1, alpha=alpha, **{n: d[n] for n in NAMES})  # fmt: skip

    out = run()
    assert torch.equal(run(), out)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    torch.testing.assert_close(out.float(), run().float(), atol=2e-7, rtol=2**-7 if kw["dtype"] == BF else 2**-10)
    ref = O.hstu_paged_forward(c["q"], c["k"], c["v"], c["kv_cache"], out_dtype=torch.float32, target_group_size=1, alpha=alpha,
                               silu_scale=0.0, max_seq_len=c["max_seq_len"], max_seq_len_k=c["max_seq_len_k"],
                               **{n: c[n] for n in NAMES})  # fmt: skip
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("dim", [64, 128])
def test_fp8(dim, monkeypatch):
    rows, keys = [1, 100, 128, 40], [2500, 3000, 2100, 2049]
    gen = torch.Generator().manual_seed(dim)
    q, k, v = ((torch.randn(n, 2, dim, generator=gen) * 0.5).to(torch.float8_e4m3fn) for n in (sum(rows), sum(keys), sum(keys)))
    kw = dict(max_seq_len=128, max_seq_len_k=3000, silu_scale=1 / 128, seq_offset=offsets(rows).to(DEV), seq_offset_k=offsets(keys).to(DEV),
              alpha=dim**-0.5)  # fmt: skip
    out = ops_rec.hstu_jagged_fp8(q.to(DEV), k.to(DEV), v.to(DEV), **kw)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    whole = ops_rec.hstu_jagged_fp8(q.to(DEV), k.to(DEV), v.to(DEV), **kw)
    torch.testing.assert_close(out.float(), whole.float(), atol=2e-7, rtol=2**-7)
    ref = O.hstu_jagged_forward(q.float(), k.float(), v.float(), out_dtype=torch.float32,
                                **dict(kw, seq_offset=offsets(rows), seq_offset_k=offsets(keys)))  # fmt: skip
    # P is rounded to e4m3 (2^-4 of a value) before it is summed over thousands of keys: far below half a step of the sum's scale
    torch.testing.assert_close(out.float().cpu(), ref, atol=2**-5 * float(ref.abs().max()), rtol=0)
