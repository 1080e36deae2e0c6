"""The backward's order that hands dS alone from the key-tile kernel to the query-tile kernel (hstu_bwd_fused_kernel.hip.h, forced with
HSTU_MI355_BWD_HANDOFF=3): against torch autograd on the CPU oracle and the library's generic kernels (the bars of
test_gpu_backward.py, the workspace full of NaN), and against the order that recomputes everything."""

import dataclasses

import pytest
import torch

import helpers
from ops_rec import workloads
from test_gpu_backward import DEV, check, device_grads, make
from test_host_backward_best_workspace import tiles

pytestmark = pytest.mark.gpu


def grad_for(w, seed=6):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(w.q.shape[0], w.q.shape[1], w.v.shape[2], generator=g, device=DEV).to(w.q.dtype)


def bytes_of_tiles(w):
    args = helpers.backward_args(w, None)
    max_q, max_k, offs_q, offs_k, context = args[7], args[8], args[10], args[11], args[12]
    whole = w.mask_type != 0 or context is not None or offs_k is not offs_q or max_q != max_k
    return tiles(rows=w.q.shape[0], batch=offs_q.numel() - 1, heads=w.q.shape[1], blocks=(max_k + 31) // 32, below_diagonal=not whole)


def against_recomputing(w, monkeypatch):
    grad_out = grad_for(w)
    helpers.set_switch(monkeypatch, "HSTU_MI355_GENERIC_BACKWARD", "0")
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "0")
    two = device_grads(w, grad_out)
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    got, beside = helpers.allocated_beside(lambda: device_grads(w, grad_out))
    # this order ran: the other ones' workspaces are of other sizes (beside the workspace: a few counts that backward_args makes)
    assert 0 <= beside - bytes_of_tiles(w) < 2048
    # S is formed with its operands the other way round and dS is rounded before dQ's product, as before dK's: one rounding of the
    # input type in the terms of a sum
    tol = 1e-2 if w.q.dtype == torch.bfloat16 else 2e-3
    for a, b in zip(got, two):
        if b is not None and b.numel():
            torch.testing.assert_close(a.float(), b.float(), atol=tol * b.float().abs().max().item(), rtol=tol)
    if w.attn_bias is not None:
        assert torch.equal(got[3] == 0, two[3] == 0)
    return got


CASES = {
    "tile_edges": dict(batch=9, dim=128, lo=0, hi=0, lengths=[1, 31, 32, 33, 127, 128, 129, 257, 384], max_seq_len=384),
    "tile_edges_64": dict(batch=9, dim=64, lo=0, hi=0, lengths=[1, 31, 32, 33, 127, 128, 129, 257, 384], max_seq_len=384),
    "tile_edges_256": dict(batch=8, dim=256, lo=0, hi=0, lengths=[1, 31, 33, 95, 127, 129, 160, 257], max_seq_len=257),
    "loose_bound": dict(batch=5, dim=128, lo=70, hi=300, max_seq_len=1000),
    "empty_sequences": dict(batch=5, dim=64, lo=0, hi=0, lengths=[0, 200, 0, 0, 65], max_seq_len=200),
    "grouped_heads": dict(batch=3, dim=128, heads=6, heads_k=2, lo=66, hi=300, max_seq_len=300),
    "dims_40_48": dict(batch=3, dim=40, dim_v=48, heads=3, lo=66, hi=300, max_seq_len=300),
    "dims_72_128": dict(batch=3, dim=72, dim_v=128, lo=66, hi=300, max_seq_len=301),
    "dims_128_16": dict(batch=3, dim=128, dim_v=16, lo=66, hi=300, max_seq_len=300),
    "dims_200_144": dict(batch=3, dim=200, dim_v=144, lo=66, hi=300, max_seq_len=300),
    "context_targets_groups": dict(batch=4, dim=128, lo=150, hi=400, max_seq_len=400, num_context=37, max_target=50, target_group_size=3),
    "context_in_the_first_block": dict(batch=4, dim=64, lo=150, hi=400, max_seq_len=400, num_context=5, max_target=1, target_group_size=1),
    "targets": dict(batch=4, dim=256, lo=100, hi=260, max_seq_len=260, max_target=70, target_group_size=1),
    "int64_offsets": dict(batch=4, dim=64, lo=70, hi=260, max_seq_len=260, index_dtype=torch.int64),
}  # fmt: skip


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("name", list(CASES))
def test_causal(name, dtype, monkeypatch):
    kw = dict(CASES[name])
    w = make(heads=kw.pop("heads", 2), seed=len(name), dtype=dtype, **kw)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    check(w, monkeypatch)
    against_recomputing(w, monkeypatch)


BIAS_CASES = {
    "rows_of_16_bytes": dict(dim=128, lengths=[1, 31, 33, 128, 129, 255, 257, 264], max_seq_len=264),
    "rows_of_16_bytes_64": dict(dim=64, lengths=[0, 31, 33, 128, 129, 255, 257, 264], max_seq_len=264),
    "rows_of_16_bytes_256": dict(dim=256, lengths=[1, 31, 96, 129, 136], max_seq_len=136),
    "loose_bound": dict(dim=64, lengths=[40, 200, 65], max_seq_len=520),
    "rows_of_8_bytes": dict(dim=128, lengths=[300, 299, 297, 150, 37], max_seq_len=300),
    "rows_of_4_bytes": dict(dim=64, lengths=[298, 297, 291, 150, 37], max_seq_len=298),
    "rows_of_4_bytes_256": dict(dim=256, lengths=[130, 129, 125, 33], max_seq_len=130),
    "dims_48_32": dict(dim=48, dim_v=32, lengths=[90, 201], max_seq_len=202),
    "context_targets_groups": dict(dim=128, lengths=[390, 160, 301], max_seq_len=392, num_context=37, max_target=50, target_group_size=3),
    "grouped_heads": dict(dim=64, heads=4, heads_k=2, lengths=[100, 250], max_seq_len=256),
}  # fmt: skip


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("name", list(BIAS_CASES))
def test_attn_bias_and_its_gradient(name, dtype, monkeypatch):
    kw = dict(BIAS_CASES[name])
    w = make(batch=len(kw["lengths"]), heads=kw.pop("heads", 2), seed=len(name), dtype=dtype, lo=0, hi=0, rab_std=0.5, **kw)
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    check(w, monkeypatch)
    against_recomputing(w, monkeypatch)


@pytest.mark.parametrize("max_seq_len", [304, 300, 298])
def test_bias_gradient_written_by_the_line(max_seq_len, monkeypatch):
    """Two query tiles per compute unit and more: the rows of the gradient leave 64 keys at a time, the block of an odd last step on its
    own, and no store reaches into the next row."""
    lengths = [max_seq_len - i % 40 for i in range(70)]
    w = make(batch=70, heads=4, dim=64, lo=0, hi=0, lengths=lengths, max_seq_len=max_seq_len, rab_std=0.5, seed=5)
    assert w.q.shape[0] // 128 * 4 >= 2 * torch.cuda.get_device_properties(0).multi_processor_count
    helpers.poison_workspace(monkeypatch)
    against_recomputing(w, monkeypatch)


@pytest.mark.parametrize("batch,heads", [(40, 1), (67, 2), (400, 2)])
@pytest.mark.parametrize("dim", [64, 128, 256])
def test_many_small_gradients_are_cleared(batch, heads, dim, monkeypatch):
    """Clearing workgroups by the number of 32-row groups (at least 8, a multiple of 8, at most a share of the compute units): each group
    is cleared once, whatever their number."""
    w = make(batch=batch, heads=heads, dim=dim, lo=1, hi=100, max_seq_len=104, rab_std=0.5, seed=batch)
    helpers.poison_workspace(monkeypatch)
    against_recomputing(w, monkeypatch)


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("mask_type", [0, 2], ids=["causal", "none"])
@pytest.mark.parametrize("lq,lk", [([70, 200, 1, 96], [370, 333, 129, 96]), ([300, 129, 40], [65, 200, 0])], ids=["more_keys", "fewer_keys"])
def test_key_offsets_of_their_own(dim, mask_type, lq, lk, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(dim)
    mk = lambda n, d: (torch.randn(n, 2, d, generator=g, device=DEV) * 0.5).to(torch.bfloat16)  # noqa: E731
    offs = lambda ls: torch.tensor([0] + list(torch.tensor(ls).cumsum(0)), dtype=torch.int64, device=DEV)  # noqa: E731
    w = workloads.Workload(name="delta", q=mk(sum(lq), dim), k=mk(sum(lk), dim), v=mk(sum(lk), dim), seq_offset=offs(lq),
                           max_seq_len=max(lq), silu_scale=1.0, alpha=dim**-0.5, seq_offset_k=offs(lk), max_seq_len_k=max(lk), lengths=lq,
                           mask_type=mask_type)  # fmt: skip
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    check(w, monkeypatch)
    against_recomputing(w, monkeypatch)


@pytest.mark.parametrize("heads_k", [4, 2], ids=["own", "grouped"])
def test_heads_over_several_launches(heads_k, monkeypatch):
    """With room for some of the heads the tiles are used by one share of them after the other: the same bits."""
    w = make(batch=5, heads=4, heads_k=heads_k, dim=64, lo=100, hi=600, max_seq_len=600, seed=3)
    grad_out = grad_for(w)
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_WORKSPACE_MB", None)
    whole, room = helpers.allocated_beside(lambda: device_grads(w, grad_out))
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_WORKSPACE_MB", str(room // 2 // 2**20 + 1))
    helpers.poison_workspace(monkeypatch)
    shares, less = helpers.allocated_beside(lambda: device_grads(w, grad_out))
    assert 0 < less <= 0.6 * room
    assert all(torch.equal(a, b) for a, b in zip(whole[:3], shares[:3]))


@pytest.mark.parametrize("dim", [64, 128, 256])
def test_rows_and_keys_that_belong_to_no_tile(dim, monkeypatch):
    """Rows ahead of the first offset and past max_seq_len are not written, rows past the last offset are zero, and a row of dO that is
    infinite reaches the keys it sees and no tile that it does not."""
    w = make(batch=3, heads=2, dim=dim, lo=200, hi=260, max_seq_len=260, seed=4)
    grad_out = grad_for(w)
    row = int(w.seq_offset[1]) + 70  # a row of the second sequence: its keys 0 .. 70
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    clean = device_grads(w, grad_out)
    bad = grad_out.clone()
    bad[row, 0] = float("inf")
    dirty = device_grads(dataclasses.replace(w), bad)
    first = int(w.seq_offset[1])
    for a, b in zip(clean[1:3], dirty[1:3]):
        assert not torch.isfinite(b[first : first + 64, 0]).all()
        keep = torch.ones(a.shape[0], dtype=torch.bool, device=DEV)
        keep[first : first + 96] = False  # (the 32-key blocks that the row's 32-row block touches)
        assert torch.equal(a[keep], b[keep]) and torch.equal(a[:, 1], b[:, 1])


@pytest.mark.parametrize("max_q,max_k", [(160, 260), (260, 160), (200, 200)])
def test_sequences_longer_than_the_bounds(max_q, max_k, monkeypatch):
    """Sequences are cut at either bound, and a causal mask is aligned to their ends: with fewer rows than keys kept, rows see past the
    diagonal.  Rows and keys past the bounds are not written."""
    w = make(batch=0, heads=2, dim=64, lo=0, hi=0, lengths=[250, 260, 90, 255], max_seq_len=260, seed=4)
    w.seq_offset_k, w.max_seq_len, w.max_seq_len_k = w.seq_offset, max_q, max_k
    grad_out = grad_for(w)
    got = {}
    for order in ("0", "1", "2", "3"):
        helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", order)
        got[order] = device_grads(w, grad_out)
    for i, bound in enumerate((max_q, max_k, max_k)):
        for b, n in enumerate(w.lengths):
            first = int(w.seq_offset[b])
            rows = slice(first, first + min(n, bound))
            want = got["0"][i][rows].float()
            for order in ("1", "2", "3"):
                torch.testing.assert_close(got[order][i][rows].float(), want, atol=1e-2 * want.abs().max().item(), rtol=1e-2)
