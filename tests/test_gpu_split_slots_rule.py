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


def params(batch, heads, heads_k, dim, rows, keys, dtype=BF, dim_v=None, context=False, bias=False):
    p = _native.new_params()
    p.q, p.k, p.v, p.out, p.seq_offset_q, p.seq_offset_k = (0x100000 * i for i in range(1, 7))  # never dereferenced
    p.dtype = _native.DT_FP8_E4M3 if dtype == F8 else _native.DT_BF16
    p.out_dtype = _native.DT_BF16
    p.n_offsets, p.num_heads_q, p.num_heads_k, p.head_dim_qk, p.head_dim_v = batch + 1, heads, heads_k, dim, dim_v or dim
    p.max_seq_len_q, p.max_seq_len_k, p.total_q, p.total_k = rows, keys, batch * rows, batch * keys
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


@pytest.mark.parametrize("case", list(test_gpu_split_slots.CASES))
def test_the_results_are_checked_on_the_slots(case, monkeypatch):
    kw, rows, keys, _ = test_gpu_split_slots.CASES[case]
    targets = kw.get("max_target", 0)  # (up to so many rows and keys more)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "1")
    max_q, max_k = max(rows) + targets, max(keys) + (max(rows) if targets else 0)
    name = name_of(params(len(rows), kw["heads"], kw.get("heads_k", kw["heads"]), kw["dim"], max_q, max_k, dim_v=kw.get("dim_v")))
    assert name.endswith("_slots_split"), name
