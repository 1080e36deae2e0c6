"""Grids of more slots than the kernel for short work lists takes: the call goes to the lists, with and without HSTU_MI355_SHORT=1 (nothing is
launched: the addresses are not any tensor's)."""

import ctypes

import pytest

import helpers
from ops_rec import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("forced", [None, "1"])
@pytest.mark.parametrize("dim,keys", [(32, 512), (64, 1024), (128, 1024)])
@pytest.mark.parametrize("max_q,short", [(16384, True), (16385, False)])
def test_slots(max_q, short, dim, keys, forced, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", forced)
    p = _native.new_params()
    p.q, p.k, p.v, p.out, p.seq_offset_q, p.seq_offset_k = (0x100000 * i for i in range(1, 7))
    p.dtype = p.out_dtype = _native.DT_BF16
    p.n_offsets, p.num_heads_q, p.num_heads_k, p.head_dim_qk, p.head_dim_v = 2049, 16, 16, dim, dim
    p.max_seq_len_q, p.max_seq_len_k, p.total_q, p.total_k = max_q, keys, 2048 * max_q, 2048 * 10
    p.alpha, p.silu_scale = 0.125, 1.0
    name = _native.load().hstu_jagged_fwd_kernel_name(ctypes.byref(p))
    assert name is not None, _native.last_error()
    by_rule = dim > 32  # (at the slot 32 lists as long as this are the queues')
    assert name.decode().endswith("_short") == (short and (by_rule or forced is not None)), name
