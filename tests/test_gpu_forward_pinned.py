"""The forward with the output sums in pinned accumulators (hstu_fwd_pinned_kernel.hip.h; host rule: 16-bit inputs, no bias, no custom mask, more
slots than a launch without a list takes, mean lengths of at least half the largest; at the slot 128 long histories only).

Every case is compared with the same sequences run in batches small enough for hstu_fwd_kernel without a list, and with the CPU oracle.  The
two kernels round the same values and add the same products in the same order: the outputs are the same bits.
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
EDGES = [1, 31, 32, 33, 64, 127, 128, 129, 160, 255, 256, 257, 300, 0, 290, 298, 300]


def prepared(w):
    k_offs = w.seq_offset if w.seq_offset_k is None else w.seq_offset_k
    max_k = w.max_seq_len if w.max_seq_len_k is None else w.max_seq_len_k
    return _ops.prepare_forward(w.q, w.k, w.v, None, None, w.mask_type, w.max_seq_len, max_k, w.silu_scale, w.seq_offset, k_offs,
                                w.num_context, w.num_target, w.target_group_size, w.alpha)  # fmt: skip


def part_of(w, b0, b1):
    """Sequences b0 .. b1 - 1 of workload w, and their query rows."""
    ko = w.seq_offset if w.seq_offset_k is None else w.seq_offset_k
    q0, q1, k0, k1 = int(w.seq_offset[b0]), int(w.seq_offset[b1]), int(ko[b0]), int(ko[b1])
    pick = lambda t: None if t is None else t[b0:b1].contiguous()  # noqa: E731
    p = workloads.Workload(name="part", q=w.q[q0:q1], k=w.k[k0:k1], v=w.v[k0:k1], seq_offset=(w.seq_offset[b0 : b1 + 1] - q0).contiguous(),
                           max_seq_len=w.max_seq_len, silu_scale=w.silu_scale, alpha=w.alpha, mask_type=w.mask_type,
                           num_context=pick(w.num_context), num_target=pick(w.num_target), target_group_size=w.target_group_size,
                           lengths=[])  # fmt: skip
    if w.seq_offset_k is not None:
        p.seq_offset_k, p.max_seq_len_k = (ko[b0 : b1 + 1] - k0).contiguous(), w.max_seq_len_k
    return p, (q0, q1)


CASES = {
    "edges": (dict(lengths=EDGES * 5, heads=2, dim=256), BF),
    "edges, fp16": (dict(lengths=EDGES * 5, heads=2, dim=256), FP),
    "grouped heads": (dict(lengths=EDGES * 3, heads=6, heads_k=2, dim=256), BF),
    "odd number of pairs, dims between slots": (dict(lengths=EDGES * 6 + [300], heads=1, dim=200, dim_v=144), BF),
    "wider values": (dict(lengths=EDGES * 5, heads=2, dim=72, dim_v=240), BF),
    "context and targets": (dict(lengths=[n + 41 for n in EDGES] * 5, heads=2, dim=256, num_context=5, max_target=40, target_group_size=3), BF),
    "long context": (dict(lengths=[300, 150, 280] * 16, heads=2, dim=256, num_context=130, max_target=9), FP),
    "no mask": (dict(lengths=EDGES * 5, heads=2, dim=256, mask_type=2), BF),
    "many short": (dict(lengths=[70, 128, 65, 100] * 70, heads=1, dim=256), FP),
    "64-bit offsets": (dict(lengths=EDGES * 5, heads=2, dim=256, index_dtype=torch.int64), BF),
    "history": (dict(lengths=[130, 129, 256, 200] * 18, heads=2, dim=256, history=500), BF),
    "history, grouped": (dict(lengths=[130, 31, 256, 200] * 15, heads=4, heads_k=2, dim=256, history=450), FP),
    "history, four tiles a pair": (dict(lengths=[400, 130, 500, 290] * 12, heads=2, dim=256, history=600), BF),
    "fewer keys than rows": (dict(lengths=[130, 129, 256, 200] * 18, heads=2, dim=256, history=-60), BF),
}


@pytest.mark.parametrize("name", list(CASES))
def test_against_the_kernel_without_a_list_and_the_oracle(name):
    kw, dtype = CASES[name]
    kw = dict(kw)
    history, mask_type = kw.pop("history", 0), kw.pop("mask_type", 0)
    w = workloads.make(name, batch=len(kw["lengths"]), lo=0, hi=0, dtype=dtype, std=0.5, seed=len(name), **kw)
    w.mask_type = mask_type
    gen = torch.Generator().manual_seed(3)
    rand = lambda rows, heads, dim: (torch.randn(rows, heads, dim, generator=gen) * 0.5).to(dtype)  # noqa: E731
    if history:
        lk = [max(0, n + history) for n in kw["lengths"]]
        w.seq_offset_k = torch.tensor([0] + lk).cumsum(0).to(w.seq_offset.dtype)
        w.max_seq_len_k = max(lk)
        w.k, w.v = (rand(sum(lk), w.k.shape[1], t.shape[2]) for t in (w.k, w.v))
    d = w.to(DEV)
    d.q = torch.cat([d.q, torch.randn(3, d.q.shape[1], d.q.shape[2], device=DEV).to(dtype)])  # rows past the last offset
    p = prepared(d)
    assert p.kernel_name().endswith("_pinned"), p.kernel_name()
    out = p.launch()
    assert not out[-3:].any()
    ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
    scale = float(ref.abs().max())
    torch.testing.assert_close(out[:-3].float().cpu(), ref, atol=(2**-6 if dtype == BF else 2**-8) * scale, rtol=2**-7)
    batch = len(kw["lengths"])
    for b0 in range(0, batch, 12):
        part, (q0, q1) = part_of(d, b0, min(b0 + 12, batch))
        if q1 == q0:
            continue
        pp = prepared(part)
        assert not pp.kernel_name().endswith("_pinned"), pp.kernel_name()
        same = pp.launch()
        assert torch.equal(out[q0:q1], same)


@pytest.mark.parametrize(
    "heads,heads_k,dim,dim_v,dtype,extra",
    [
        (2, 2, 128, 128, BF, dict()),
        (4, 2, 128, 128, BF, dict(num_context=3, max_target=40, target_group_size=3)),
        (2, 2, 128, 128, FP, dict(index_dtype=torch.int64)),
        (3, 3, 96, 80, BF, dict()),
    ],
    ids=str,
)
def test_histories_at_the_slot_128(heads, heads_k, dim, dim_v, dtype, extra, monkeypatch):
    batch = 210
    lengths = [129, 200, 161, 256, 255, 130, 200] * (batch // 7)
    w = workloads.make("history", batch=batch, heads=heads, heads_k=heads_k, dim=dim, dim_v=dim_v, lo=0, hi=0, lengths=lengths, dtype=dtype,
                       std=0.5, seed=dim, device=DEV, **extra)  # fmt: skip
    lk = [1350 + 37 * (i % 9) for i in range(batch)]
    w.seq_offset_k = torch.tensor([0] + lk, device=DEV).cumsum(0).to(w.seq_offset.dtype)
    w.max_seq_len_k = max(lk)
    w.k, w.v = (torch.randn(sum(lk), heads_k, t.shape[2], device=DEV).mul_(0.5).to(dtype) for t in (w.k, w.v))
    out = prepared(w)
    assert out.kernel_name().endswith("_d128_rabfalse_maskfalse_pinned"), out.kernel_name()
    out = out.launch()
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    for b0 in range(0, batch, 30):
        part, (q0, q1) = part_of(w, b0, b0 + 30)
        pp = prepared(part)
        assert not pp.kernel_name().endswith("_pinned"), pp.kernel_name()
        same = pp.launch()
        assert torch.equal(out[q0:q1], same)


def test_every_replay_of_a_captured_launch_is_the_eager_result():
    w = workloads.make("capture", batch=40, heads=4, dim=256, lo=200, hi=300, dtype=BF, device=DEV, seed=2)
    p = prepared(w)
    assert p.kernel_name().endswith("_pinned")
    want = p.launch().clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = p.launch()
    for _ in range(4):
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_the_switch_for_the_persistent_kernel(monkeypatch):
    w = workloads.make("switch", batch=40, heads=4, dim=256, lo=200, hi=300, dtype=FP, device=DEV, seed=2)
    p = prepared(w)
    assert p.kernel_name().endswith("_pinned")
    out = p.launch()
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    p = prepared(w)
    assert not p.kernel_name().endswith("_pinned")
    assert torch.equal(p.launch(), out)


def test_batches_the_rule_leaves_to_the_lists():
    def name(**kw):
        w = workloads.make("route", batch=kw.pop("batch", 40), dtype=BF, device=DEV, seed=1, **kw)
        d_bias = w.attn_bias
        return _ops.prepare_forward(w.q, w.k, w.v, None, d_bias, 0, w.max_seq_len, w.max_seq_len, w.silu_scale, w.seq_offset, w.seq_offset,
                                    None, None, 0, w.alpha).kernel_name()  # fmt: skip

    assert name(heads=4, dim=256, lo=200, hi=300).endswith("_pinned")
    assert name(heads=4, dim=128, lo=200, hi=1100).find("_pinned") < 0
    assert name(heads=4, dim=256, lo=200, hi=300, rab_std=0.2).find("_pinned") < 0
    assert name(heads=4, dim=256, lo=200, hi=300, max_seq_len=800).find("_pinned") < 0  # most slots would be empty
    assert name(heads=4, dim=256, lo=200, hi=300, batch=8).endswith("_direct")
    for batch, taken in ((26, False), (60, True)):  # on a history, a tile per compute unit at most: 2 x 4 x 26 with rows of 100 .. 300
        w = workloads.make("route", batch=batch, heads=4, dim=256, lo=0, hi=0, lengths=[100, 300] * (batch // 2), dtype=BF, device=DEV)
        w.seq_offset_k = torch.arange(0, 601 * batch, 600, device=DEV)[: batch + 1].to(w.seq_offset.dtype)
        w.max_seq_len_k = 600
        w.k = w.v = torch.zeros(600 * batch, 4, 256, dtype=BF, device=DEV)
        assert prepared(w).kernel_name().endswith("_pinned") == taken


@pytest.mark.parametrize(
    "batch,heads,heads_k,dim,rows,keys,kernel",
    [
        (200, 2, 2, 128, (400, 400), 3072, "_pinned"),
        (100, 8, 8, 128, (400, 400), 2256, "_queues"),  # six items per resident workgroup: the queues take them pair after pair
        (100, 8, 4, 128, (400, 400), 3072, "_queues"),
        (120, 4, 4, 128, (185, 698), 3000, "_pinned"),  # uneven rows: pair after pair from four items on
        (165, 4, 4, 128, (185, 698), 3000, "_queues"),
        (400, 2, 2, 128, (400, 400), 1000, "_pinned"),  # as many items, but the kernel for short lists would take them
        (22, 4, 4, 128, (1100, 1100), 7000, "_split"),  # a few workgroups in a second round of long sweeps
        (31, 4, 4, 128, (1100, 1100), 7000, "_pinned"),
        (134, 2, 2, 128, (218, 592), 2584, "_d128_rabfalse_maskfalse"),  # uneven rows: the lists sort them
        (190, 2, 2, 128, (218, 592), 2584, "_pinned"),
        (124, 8, 8, 128, (80, 140), 1000, "_short"),  # half of the second tiles missing
        (124, 8, 8, 128, (120, 200), 1000, "_pinned"),
        (12, 2, 2, 256, (2000, 3000), 7000, "_d256_rabfalse_maskfalse"),  # few rounds of long sweeps
        (13, 2, 2, 256, (2000, 3000), 7000, "_pinned"),
        (17, 4, 2, 256, (700, 1000), 4500, "_d256_rabfalse_maskfalse"),
        (20, 4, 2, 256, (700, 1000), 4500, "_pinned"),
        (5, 4, 4, 256, (3500, 3500), 8000, "_d256_rabfalse_maskfalse"),  # fewer than three pairs per XCD
        (10, 4, 4, 256, (3500, 3500), 8000, "_pinned"),
    ],
)
def test_histories_that_the_lists_order_better(batch, heads, heads_k, dim, rows, keys, kernel):
    lo, hi = rows
    lengths = [lo + (hi - lo) * (2 * i + 1) // (2 * batch) for i in range(batch)]
    q = torch.empty(sum(lengths), heads, dim, dtype=BF, device=DEV)
    kv = torch.empty(keys * batch, heads_k, dim, dtype=BF, device=DEV)
    offsets = torch.tensor([0] + lengths, device=DEV).cumsum(0).to(torch.int32)
    offsets_k = torch.arange(0, keys * batch + 1, keys, device=DEV, dtype=torch.int32)
    name = _ops.prepare_forward(q, kv, kv, None, None, 0, hi, keys, 1.0, offsets, offsets_k, None, None, 0, 1.0).kernel_name()
    assert name.removesuffix("_split").endswith(kernel.removesuffix("_split")), name
