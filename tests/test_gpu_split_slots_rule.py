"""Which rows on a history run in slots that cut all items alike, and which from a list, paged and not: both sides of each line of the rule on 256
compute units (nothing is launched).  The cases of test_gpu_split_slots.py are all on the slots' side."""

import ctypes

import pytest
import torch

import helpers
import test_gpu_split_slots
from ops_rec import _native

pytestmark = pytest.mark.gpu
BF, F8 = torch.bfloat16, torch.float8_e4m3fn


def params(batch, heads, heads_k, dim, rows, keys, dtype=BF, dim_v=None, context=False, bias=False, mean=None):
    p = _native.new_params()
    p.q, p.k, p.v, p.out, p.seq_offset_q, p.seq_offset_k = (0x100000 * i for i in range(1, 7))  # never dereferenced
    p.dtype = _native.DT_FP8_E4M3 if dtype == F8 else _native.DT_BF16
    p.out_dtype = _native.DT_BF16
    p.n_offsets, p.num_heads_q, p.num_heads_k, p.head_dim_qk, p.head_dim_v = batch + 1, heads, heads_k, dim, dim_v or dim
    p.max_seq_len_q, p.max_seq_len_k, p.total_q, p.total_k = rows, keys, batch * (mean or rows), batch * keys
    p.alpha, p.silu_scale = 0.125, 1.0
    p.num_context = 0x800000 if context else None
    p.attn_bias = 0x900000 if bias else None
    return p


def name_of(p, paged=False):
    lib = _native.load()
    if paged:
        pp = _native.PagedParams()
        pp.struct_size = ctypes.sizeof(_native.PagedParams)
        pp.fwd = p
        pp.kv_cache, pp.page_offsets, pp.page_ids, pp.last_page_len, pp.seq_offset_t = (0x1000000 * i for i in range(1, 6))
        pp.num_pages, pp.page_size, pp.n_page_ids = 100, 128, 100
        name = lib.hstu_paged_fwd_kernel_name(ctypes.byref(pp))
    else:
        name = lib.hstu_jagged_fwd_kernel_name(ctypes.byref(p))
    assert name is not None, _native.last_error()
    return name.decode()


@pytest.mark.parametrize(
    "args,kw,ending",
    [
        ((4, 2, 2, 128, 128, 600), dict(), "_slots_split"),
        ((4, 2, 2, 128, 128, 600), dict(context=True), "_maskfalse_split"),
        ((4, 2, 2, 128, 128, 600), dict(bias=True), "_rabtrue_maskfalse_split"),
        ((4, 2, 2, 64, 300, 600), dict(), "_slots_split"),  # several tiles: as many keys behind the rows as there are rows
        ((4, 2, 2, 64, 301, 600), dict(), "_maskfalse_split"),
        ((64, 4, 4, 128, 100, 600), dict(), "_slots_split"),  # 256 pairs, two parts each
        ((257, 1, 1, 128, 100, 600), dict(), "_maskfalse_split"),
        ((64, 4, 2, 128, 200, 600), dict(), "_maskfalse_split"),  # 128 pairs of four workgroups
        ((32, 4, 2, 128, 200, 600), dict(), "_slots_split"),
        ((384, 1, 1, 64, 100, 600), dict(), "_slots_split"),
        ((385, 1, 1, 64, 100, 600), dict(), "_maskfalse_split"),
        ((384, 1, 1, 64, 100, 2000), dict(dtype=F8), "_slots_split"),
        ((385, 1, 1, 64, 100, 2000), dict(dtype=F8), "_d64_split"),
        ((4, 2, 2, 256, 100, 1025), dict(), "_slots_split"),
        ((4, 2, 2, 256, 100, 1024), dict(), "_direct"),
        ((128, 1, 1, 256, 100, 2000), dict(), "_slots_split"),
        ((129, 1, 1, 256, 100, 2000), dict(), "_direct"),
        ((4, 2, 2, 256, 300, 600), dict(), "_direct"),
        ((4, 2, 2, 32, 128, 2000), dict(), "_direct"),
    ],
    ids=str,
)
def test_rows_on_a_history(args, kw, ending, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "1")
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    name = name_of(params(*args, **kw))
    assert name.endswith(ending), name


@pytest.mark.parametrize(
    "args,kw,ending",
    [
        ((4, 2, 2, 128, 100, 300), dict(), "_slots_paged"),  # whole items
        ((512, 1, 1, 128, 100, 300), dict(), "_slots_paged"),
        ((513, 1, 1, 128, 100, 300), dict(), "_maskfalse_paged"),
        ((96, 8, 8, 64, 100, 3000), dict(), "_slots_paged"),
        ((97, 8, 8, 64, 100, 3000), dict(), "_maskfalse_paged"),
        ((4, 2, 2, 128, 300, 600), dict(), "_slots_paged"),
        ((4, 2, 2, 128, 301, 600), dict(), "_maskfalse_paged"),
        ((256, 1, 1, 256, 100, 3000), dict(), "_slots_paged"),
        ((257, 1, 1, 256, 100, 3000), dict(), "_maskfalse_paged"),
        ((4, 2, 2, 256, 100, 3000), dict(bias=True), "_rabtrue_maskfalse_paged"),
        ((4, 2, 2, 32, 100, 3000), dict(), "_direct"),  # gathered
    ],
    ids=str,
)
def test_paged(args, kw, ending, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    name = name_of(params(*args, **kw), paged=True)
    assert name.endswith(ending), name


@pytest.mark.parametrize(
    "args,mean,paged,ending",
    [
        # uneven rows at the slot 128: two parts of each slot, or those that a list makes of the tiles that the mean length tells of
        ((22, 2, 1, 128, 429, 6254), 241, False, "_maskfalse_split"),  # 176 slots, 104 tiles: 4.9 parts spare 58 steps of 196
        ((22, 2, 1, 128, 429, 2080), 241, False, "_slots_split"),  # 19.2 of 65
        ((22, 2, 1, 128, 429, 6254), 414, False, "_slots_split"),  # 176 tiles: no room for a third part of each
        ((10, 4, 4, 128, 300, 7000), 80, False, "_slots_split"),  # four parts of each slot
        ((50, 2, 2, 128, 200, 3000), 150, False, "_slots_split"),  # 200 slots, 167 tiles: 16.3 steps of 94, two rounds either way
        ((50, 2, 2, 128, 200, 3700), 150, False, "_maskfalse_split"),  # 20.2 of 116
        # at the slot 64 from 25 steps on, or ten and a round less
        ((82, 2, 2, 64, 166, 2560), 110, False, "_maskfalse_split"),  # 328 slots, 223 tiles
        ((82, 2, 2, 64, 166, 1500), 110, False, "_slots_split"),  # two rounds instead of three, but 9.9 steps
        # whole items of paged calls: two parts of each tile, or a round less
        ((68, 2, 1, 128, 222, 3600), 130, True, "_maskfalse_paged"),
        ((68, 2, 1, 128, 222, 3600), 215, True, "_slots_paged"),
        ((363, 1, 1, 64, 149, 5400), 99, True, "_maskfalse_paged"),  # 462 tiles: two rounds instead of three
        ((363, 1, 1, 64, 149, 5400), 140, True, "_slots_paged"),
        ((52, 1, 1, 256, 400, 3000), 100, True, "_slots_paged"),  # no rule at the slot 256
        ((4, 2, 2, 128, 100, 6000), 20, False, "_slots_split"),  # one tile
    ],
    ids=str,
)
def test_uneven_rows(args, mean, paged, ending, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "1")
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    name = name_of(params(*args, mean=mean), paged=paged)
    assert name.endswith(ending), name


@pytest.mark.parametrize("case", list(test_gpu_split_slots.CASES))
def test_the_results_are_checked_on_the_slots(case, monkeypatch):
    kw, rows, keys, _ = test_gpu_split_slots.CASES[case]
    targets = kw.get("max_target", 0)  # (up to so many rows and keys more)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "1")
    max_q, max_k = max(rows) + targets, max(keys) + (max(rows) if targets else 0)
    name = name_of(params(len(rows), kw["heads"], kw.get("heads_k", kw["heads"]), kw["dim"], max_q, max_k, dim_v=kw.get("dim_v")))
    assert name.endswith("_slots_split"), name
