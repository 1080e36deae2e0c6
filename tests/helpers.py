"""Shared input builders for the tests (seeded, CPU)."""

from __future__ import annotations

import numpy as np
import torch

from ops_rec import workloads


def set_switch(monkeypatch, name, value):
    """Sets (``value`` a string) or unsets (None) one of the library's ``HSTU_MI355_*`` switches for the rest of the
    test: the library reads its switches from the environment once per process, so it is told to read them again.
    (``tests/conftest.py`` has it read them once more when the test's environment has been put back.)"""
    from ops_rec import _native

    if value is None:
        monkeypatch.delenv(name, raising=False)
    else:
        monkeypatch.setenv(name, value)
    _native.reload_switches()


def poison_workspace(monkeypatch):
    """Everything the operators allocate from here on -- the backward's workspace, outputs, gradients -- is handed out holding
    NaN in every element, so that a read of something never written, or an element of a result that nobody wrote, shows: torch's
    own setting, which the native kernels follow.  (``tests/conftest.py`` switches it off again.)"""
    monkeypatch.setattr(torch.utils.deterministic, "fill_uninitialized_memory", True)
    torch.use_deterministic_algorithms(True, warn_only=True)


def allocated_beside(call):
    """``call()``, and how many bytes it had asked torch's allocator for at its peak beside what it returned: the workspace of an
    operator whose arguments are taken as they are."""
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    out = call()
    stats = torch.cuda.memory_stats()
    return out, stats["requested_bytes.all.peak"] - stats["requested_bytes.all.current"]


def with_room_for(call, n_bytes, like):
    """``call()`` while torch's allocator may take no more than ``n_bytes`` from the device beyond free blocks of the sizes in
    ``like`` (its results), and how many requests it refused."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    limit = lambda n: torch.cuda.set_per_process_memory_fraction(n / total)  # noqa: E731
    blocks = [torch.empty_like(t) for t in like if t is not None]
    taken = []
    try:
        limit(torch.cuda.memory_reserved())
        for size in (1 << n for n in range(34, 19, -1)):  # (whatever is free inside blocks that live tensors keep from being given back)
            try:
                while True:
                    taken.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.cuda.OutOfMemoryError:
                pass
        del blocks
        limit(torch.cuda.memory_reserved() + n_bytes)
        before = torch.cuda.memory_stats()["num_ooms"]
        out = call()
        torch.cuda.synchronize()
        return out, torch.cuda.memory_stats()["num_ooms"] - before
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        del taken


def backward_args(w, grad):
    """The arguments of ``hstu_jagged_backward`` (its longer form) for a workload."""
    k_offs = w.seq_offset if w.seq_offset_k is None else w.seq_offset_k
    max_k = w.max_seq_len if w.max_seq_len_k is None else w.max_seq_len_k
    ctx, tgt = w.num_context, w.num_target
    if (ctx is None) != (tgt is None):  # the backward op wants both or neither (hstu_jagged_plugin.cpp:81-84)
        zeros = torch.zeros_like(ctx if tgt is None else tgt)
        ctx, tgt = (zeros if ctx is None else ctx), (zeros if tgt is None else tgt)
    return (grad, w.q, w.k, w.v, w.mask, w.attn_bias, w.mask_type, w.max_seq_len, max_k, w.silu_scale, w.seq_offset, k_offs, ctx, tgt,
            w.target_group_size, w.alpha)  # fmt: skip


def backward_without_workspace(monkeypatch, w, grad):
    """The gradients from a caller that brings no workspace, whatever the library asks for: through the Python implementation,
    whose allocations can be replaced."""
    from ops_rec import _ops

    with monkeypatch.context() as patch:
        patch.setattr(_ops, "_new_workspace", lambda n_bytes, device: None)
        return _ops.hstu_jagged_backward_delta(*backward_args(w, grad))


def small_case(seed=0, batch=3, heads=2, dim=32, lo=1, hi=40, dtype=torch.float32, std=1.0, rab=False, custom_mask=False,
               ctx=0, max_target=0, group=0, heads_k=None, dim_v=None, delta=False, index_dtype=torch.int32,
               alpha=None):  # fmt: skip
    """A small jagged batch; with ``delta`` the K/V sequences are longer than the Q sequences."""
    w = workloads.make("t", batch=batch, heads=heads, dim=dim, lo=lo, hi=hi, dtype=dtype, std=std,
                       rab_std=(0.5 if rab else None), num_context=ctx, max_target=max_target,
                       target_group_size=group, heads_k=heads_k, dim_v=dim_v, index_dtype=index_dtype, seed=seed,
                       alpha=alpha)  # fmt: skip
    g = torch.Generator().manual_seed(seed + 7)
    if delta:
        extra = torch.randint(0, 9, (len(w.lengths),), generator=g).tolist()
        len_k = [a + b for a, b in zip(w.lengths, extra)]
        total_k = sum(len_k)
        hk = heads_k or heads
        w.k = (torch.randn(total_k, hk, dim, generator=g) * std).to(dtype)
        w.v = (torch.randn(total_k, hk, dim_v or dim, generator=g) * std).to(dtype)
        offs = [0]
        for n in len_k:
            offs.append(offs[-1] + n)
        w.seq_offset_k = torch.tensor(offs, dtype=index_dtype)
        w.max_seq_len_k = max(len_k)
        if rab:
            w.attn_bias = (torch.randn(len(len_k), heads, w.max_seq_len, w.max_seq_len_k, generator=g) * 0.5).to(dtype)
    if custom_mask:
        mk = w.max_seq_len_k if w.max_seq_len_k is not None else w.max_seq_len
        w.mask = torch.randint(0, 2, (len(w.lengths), heads, w.max_seq_len, mk), generator=g).to(dtype)
        w.mask_type = 3
    return w


def reference_style_case(batch, heads, max_len, dim, dtype, *, enable_bias=False, silu_scale=0.0, mask_type=0,
                         group=0, ctx=0, tgt=0, heads_k=None, dim_v=None, min_len=1, repeat_offset=False,
                         index_dtype=torch.int32, delta=False, alpha=1.0, seed=0):  # fmt: skip
    """Inputs with the distributions of the reference's forward tests: q/k/v ~ U(-1, 1), bias ~ U(0, 1),
    lengths uniform in [min_len, max_len] (+ context + targets for the built-in mask), every sequence with the
    same num_context / num_target, a 0/1 random tensor as custom mask, max_seq_len = the longest sequence
    (hstu_forward_v1/test/pytest/test_hstu_jagged.py:41-104 and :755-800 for the delta form)."""
    g = torch.Generator().manual_seed(seed)
    heads_k = heads_k or heads
    dim_v = dim_v or dim
    lens = torch.randint(min_len, max_len + 1, (batch,), generator=g)
    if mask_type == 0:
        lens = lens + ctx + tgt
    lens_k = lens.clone()
    if delta:
        lens_k = lens + (torch.rand(batch, generator=g) * (int(lens.max()) - lens + 1)).long()
    lq, lk = lens.tolist(), lens_k.tolist()
    max_q, max_k = max(lq), max(lk)

    def offs(ls):
        o = [0]
        for n in ls:
            o.append(o[-1] + n)
        return o

    oq, ok = offs(lq), offs(lk)
    u = lambda *s: (torch.rand(*s, generator=g) * 2 - 1).to(dtype)  # noqa: E731
    q, k, v = u(oq[-1], heads, dim), u(ok[-1], heads_k, dim), u(ok[-1], heads_k, dim_v)
    bias = torch.rand(batch, heads, max_q, max_k, generator=g).to(dtype) if enable_bias else None
    mask = None
    if mask_type == 3:
        mask = torch.randint(0, 2, (batch, heads, max_q, max_k), generator=g).to(dtype)
    n_ctx = torch.full((batch,), ctx, dtype=index_dtype)
    n_tgt = torch.full((batch,), tgt, dtype=index_dtype)
    if repeat_offset:
        oq, ok = oq + oq[-1:], ok + ok[-1:]
        n_ctx, n_tgt = torch.cat([n_ctx, n_ctx[-1:]]), torch.cat([n_tgt, n_tgt[-1:]])
        if bias is not None:
            bias = torch.cat([bias, bias[-1:]])
        if mask is not None:
            mask = torch.cat([mask, mask[-1:]])
    return workloads.Workload(
        name="ref-style", q=q, k=k, v=v, seq_offset=torch.tensor(oq, dtype=index_dtype), max_seq_len=max_q,
        silu_scale=silu_scale, alpha=alpha, attn_bias=bias, mask=mask, mask_type=mask_type, num_context=n_ctx,
        num_target=n_tgt, target_group_size=group,
        seq_offset_k=(torch.tensor(ok, dtype=index_dtype) if delta else None), max_seq_len_k=(max_k if delta else None),
        lengths=lq,
    )  # fmt: skip


def paged_case(hist, prev, targets, page_size, heads=2, heads_k=None, dim=32, dtype=torch.float32, std=1.0, seed=0,
               index_dtype=torch.int32, shuffle_pages=True, spare_pages=2):
    """Inputs of ``hstu_paged`` in the way the reference's test builds them
    (hstu_forward_v1/test/pytest/test_hstu_paged.py:274-330): per sequence ``hist[b]`` new history tokens and
    ``targets[b]`` target tokens are the query rows; the cache holds ``prev[b] + hist[b]`` rows in pages of
    ``page_size``; physical pages are numbered in a shuffled order with unused spare pages in between."""
    g = torch.Generator().manual_seed(seed)
    heads_k = heads_k or heads
    batch = len(hist)
    q_lens = [h + t for h, t in zip(hist, targets)]
    k_lens = [p + h + t for p, h, t in zip(prev, hist, targets)]
    total = sum(q_lens)
    rnd = lambda *shape: (torch.randn(*shape, generator=g) * std).to(dtype)  # noqa: E731
    q, k, v = rnd(total, heads, dim), rnd(total, heads_k, dim), rnd(total, heads_k, dim)
    cached = [p + h for p, h in zip(prev, hist)]
    pages_per_seq = [(c + page_size - 1) // page_size for c in cached]
    n_pages = sum(pages_per_seq) + spare_pages
    order = torch.randperm(n_pages, generator=g).tolist() if shuffle_pages else list(range(n_pages))
    kv_cache = rnd(n_pages, 2, page_size, heads_k, dim)
    page_ids = order[: sum(pages_per_seq)]
    offs = lambda ls: torch.tensor([0] + list(np.cumsum(ls)), dtype=index_dtype)  # noqa: E731
    last = [c % page_size if c % page_size else (page_size if c else 0) for c in cached]
    return dict(
        q=q, k=k, v=v, kv_cache=kv_cache, seq_offset=offs(q_lens), seq_offset_k=offs(k_lens),
        seq_offset_t=offs(targets), page_offsets=offs(pages_per_seq), page_ids=torch.tensor(page_ids, dtype=index_dtype),
        last_page_len=torch.tensor(last, dtype=index_dtype), num_target=torch.tensor(targets, dtype=index_dtype),
        max_seq_len=max(q_lens), max_seq_len_k=max(k_lens),
    )  # fmt: skip
