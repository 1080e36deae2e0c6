"""hstu_jagged_bwd_best_workspace_size (no GPU needed): 2 KiB per head and 32 x 32 block of dS where the call takes the order that hands
dS alone over, and what hstu_jagged_bwd_workspace_size says elsewhere."""

import ctypes

import pytest

import helpers
from ops_rec import _native
from test_host_boundary import _copy_fwd, _valid_params

FAKE = 0x1000
BATCH = dict(n_offsets=33, num_heads_q=4, num_heads_k=4, total_q=20292, total_k=20292, max_seq_len_q=1024, max_seq_len_k=1024)


def sizes(grad_attn_bias=None, **fwd):
    b = _native.new_bwd_params()
    f = _valid_params()
    for k, v in fwd.items():
        setattr(f, k, v)
    if grad_attn_bias is not None:
        f.attn_bias = FAKE
    _copy_fwd(b.fwd, f)
    b.grad = b.grad_q = b.grad_k = b.grad_v = FAKE
    b.grad_attn_bias = grad_attn_bias
    ws = (ctypes.c_uint64 * 2)()
    for i, size in enumerate((_native.load().hstu_jagged_bwd_workspace_size, _native.load().hstu_jagged_bwd_best_workspace_size)):
        assert size(ctypes.byref(b), ctypes.cast(ctypes.byref(ws, 8 * i), ctypes.POINTER(ctypes.c_uint64))) == 0, _native.last_error()
    return tuple(ws)


def tiles(rows=20292, batch=32, heads=4, blocks=32, below_diagonal=True):
    groups = rows // 32 + batch
    return heads * 2048 * ((groups * (blocks + 1) + 1) // 2 if below_diagonal else groups * blocks)


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in ("HSTU_MI355_BWD_HANDOFF", "HSTU_MI355_BWD_WORKSPACE_MB", "HSTU_MI355_SHORT", "HSTU_MI355_GENERIC_BACKWARD"):
        helpers.set_switch(monkeypatch, name, None)


@pytest.mark.parametrize("dim", [64, 128, 256])
def test_tiles(dim):
    call = dict(BATCH, head_dim_qk=dim, head_dim_v=dim)
    assert sizes(**call)[1] == tiles()
    assert sizes(**dict(call, mask_type=2))[1] == tiles(below_diagonal=False)
    assert sizes(**dict(call, num_context=FAKE))[1] == tiles(below_diagonal=False)
    assert sizes(**dict(call, seq_offset_k=FAKE + 64))[1] == tiles(below_diagonal=False)
    assert sizes(**dict(call, max_seq_len_k=900))[1] == tiles(blocks=29, below_diagonal=False)  # (more query rows than keys in a sequence)
    # a sequence of more than 900 rows keeps 900 of them and up to 1024 keys: rows see keys past the diagonal
    assert sizes(**dict(call, max_seq_len_q=900))[1] == tiles(below_diagonal=False)


def test_as_the_other_orders_elsewhere():
    for call in (dict(BATCH, head_dim_qk=512, head_dim_v=512), dict(BATCH, dtype=_native.DT_FP32, out_dtype=_native.DT_FP32),
                 dict(BATCH, total_q=600, total_k=600, max_seq_len_q=32, max_seq_len_k=32),
                 dict(BATCH, n_offsets=3, total_q=500, total_k=500, max_seq_len_q=300, max_seq_len_k=300),  # a few workgroups
                 dict(BATCH, n_offsets=5, total_q=2000, total_k=2000, num_heads_k=1)):  # fmt: skip
        size, best = sizes(**call)
        assert size == best


def test_limits_and_switches(monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_WORKSPACE_MB", "60")
    size, best = sizes(**BATCH)  # room for two of the four heads, whose share of the launch would leave the machine half empty
    assert size == best
    long = dict(BATCH, n_offsets=65, total_q=64 * 4096, total_k=64 * 4096, max_seq_len_q=4096, max_seq_len_k=4096)
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_WORKSPACE_MB", "3000")
    assert sizes(**long)[1] == tiles(rows=64 * 4096, batch=64, blocks=128, heads=2)  # two pairs of launches of two heads
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_WORKSPACE_MB", None)
    for order in ("0", "1", "2"):
        helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", order)
        size, best = sizes(**BATCH)
        assert size == best
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "3")
    assert sizes(**dict(BATCH, n_offsets=3, total_q=500, total_k=500))[1] == tiles(rows=500, batch=2)


BIASED = [  # heads, K/V heads, head dim, batch, rows, bound of rows, keys; whether the call takes the dS tiles
    (8, 2, 128, 16, 640, 1024, 640, False),  # grouped heads: fewer (tiles x mean rows / longest rows) than 9/8 of the compute units
    (8, 1, 128, 32, 1024, 1024, 1024, False),
    (8, 4, 128, 32, 640, 1024, 640, True),
    (8, 2, 128, 4, 300, 300, 700, False),  # on a history: fewer tiles than half of them
    (8, 2, 128, 16, 256, 256, 1024, True),
    (2, 2, 128, 512, 114, 128, 114, False),  # rows of one tile
    (4, 4, 128, 512, 128, 128, 128, True),
    (4, 4, 128, 16, 400, 500, 400, False),  # a head each: short rows
    (4, 4, 128, 8, 768, 1024, 768, True),
    (4, 4, 128, 128, 250, 300, 250, True),
    (4, 4, 128, 32, 64, 64, 1000, True),
    (8, 2, 64, 16, 300, 400, 300, False),
    (8, 1, 64, 4, 768, 1024, 768, False),
    (8, 1, 64, 16, 640, 1024, 640, True),
    (4, 2, 64, 8, 300, 400, 300, True),
    (8, 2, 256, 4, 1536, 2048, 1536, False),
    (8, 2, 256, 16, 640, 1024, 640, True),
    (4, 2, 256, 8, 768, 1024, 768, True),
    (4, 2, 64, 8, 112, 112, 112, False),  # in pairs: short rows in at most a slot per compute unit
    (4, 2, 64, 128, 112, 112, 112, True),
    (4, 2, 64, 4, 256, 256, 256, True),
    (4, 2, 256, 26, 200, 200, 200, False),
    (4, 2, 256, 40, 200, 200, 200, True),
    (4, 2, 256, 6, 1000, 1000, 1000, True),
    (4, 4, 128, 64, 100, 100, 376, False),  # rows of one tile on a history: a slot per compute unit and more
    (4, 4, 128, 48, 100, 100, 376, True),
    (4, 2, 128, 32, 100, 100, 200, False),
    (4, 2, 128, 32, 100, 100, 376, True),
    (4, 2, 128, 128, 100, 100, 376, False),
    (4, 4, 128, 234, 136, 216, 136, False),  # short uneven rows
    (4, 4, 128, 400, 136, 216, 136, True),
    (4, 4, 128, 180, 140, 144, 140, True),
    (4, 4, 256, 56, 64, 64, 64, False),  # short single tiles of nearly all compute units, beside the clearing workgroups
    (4, 4, 256, 48, 64, 64, 64, True),
    (4, 4, 256, 40, 128, 128, 128, True),
]


@pytest.mark.parametrize("heads,heads_k,dim,batch,rows,max_rows,keys,taken", BIASED)
def test_calls_with_a_bias(heads, heads_k, dim, batch, rows, max_rows, keys, taken):
    """Where the orders without dS tiles were measured to be the faster ones (256 compute units), the call asks for their workspace."""
    own = keys != rows
    call = dict(n_offsets=batch + 1, num_heads_q=heads, num_heads_k=heads_k, head_dim_qk=dim, head_dim_v=dim, total_q=batch * rows,
                total_k=batch * keys, max_seq_len_q=max_rows, max_seq_len_k=(keys if own else max_rows), seq_offset_k=FAKE + (64 if own else 0))  # fmt: skip
    size, best = sizes(grad_attn_bias=FAKE, **call)
    whole = tiles(rows=batch * rows, batch=batch, heads=heads, blocks=(call["max_seq_len_k"] + 31) // 32, below_diagonal=not own)
    assert best == (whole if taken else size) and whole != size


UNBIASED = [  # heads, K/V heads, head dim, batch, rows, bound of rows, keys; whether the call takes the dS tiles
    (4, 4, 128, 16, 100, 100, 100, False),  # a head each at the slot 128: short rows in few tiles
    (4, 4, 96, 15, 142, 168, 142, False),
    (4, 4, 128, 32, 256, 256, 256, True),
    (4, 4, 128, 48, 140, 140, 140, True),  # more than a slot per compute unit
    (4, 4, 128, 40, 105, 200, 105, True),
    (4, 4, 128, 8, 512, 512, 512, True),
    (4, 4, 128, 16, 200, 200, 400, True),
    (4, 4, 64, 16, 100, 100, 100, True),
    (4, 4, 256, 16, 140, 140, 140, True),
    (8, 4, 128, 32, 200, 200, 200, False),  # grouped heads: last tiles partly empty, up to two slots per compute unit
    (8, 4, 128, 35, 200, 200, 200, True),
    (8, 4, 128, 24, 256, 256, 256, True),
    (8, 4, 128, 48, 100, 100, 100, True),
    (4, 2, 64, 64, 200, 200, 200, False),
    (4, 2, 128, 64, 200, 200, 400, True),
    (4, 2, 256, 64, 200, 200, 200, True),
    (4, 2, 128, 64, 100, 100, 160, False),  # rows of one tile on keys of two
    (4, 2, 128, 80, 100, 100, 160, True),
    (4, 2, 128, 64, 100, 100, 400, True),
    (4, 2, 64, 64, 100, 100, 160, True),
]


@pytest.mark.parametrize("heads,heads_k,dim,batch,rows,max_rows,keys,taken", UNBIASED)
def test_calls_without_a_bias(heads, heads_k, dim, batch, rows, max_rows, keys, taken):
    """Where the orders without dS tiles were measured to be the faster ones (256 compute units), the call asks for their workspace."""
    own = keys != rows
    call = dict(n_offsets=batch + 1, num_heads_q=heads, num_heads_k=heads_k, head_dim_qk=dim, head_dim_v=dim, total_q=batch * rows,
                total_k=batch * keys, max_seq_len_q=max_rows, max_seq_len_k=(keys if own else max_rows), seq_offset_k=FAKE + (64 if own else 0))  # fmt: skip
    size, best = sizes(**call)
    whole = tiles(rows=batch * rows, batch=batch, heads=heads, blocks=(call["max_seq_len_k"] + 31) // 32, below_diagonal=not own)
    assert best == (whole if taken else size) and whole != size


def pair_lines(groups):
    """Lines of the pair plane that ``groups`` 32-row groups take up to the diagonal (row group g: g + 1 lines a row)."""
    return 16 * groups * (groups + 1)


@pytest.mark.parametrize("max_q,max_k", [(300, 300), (300, 160), (160, 300), (640, 64)])
def test_the_planes_hold_sequences_that_are_cut(max_q, max_k, monkeypatch):
    """Sequences longer than a bound are cut at it: whatever the bounds, the plane has room for what the kernels write (the last sequence's
    lines end inside it), up to the diagonal only where rows and keys are cut alike."""
    helpers.set_switch(monkeypatch, "HSTU_MI355_BWD_HANDOFF", "2")
    heads, lengths = 2, [700, 650, 700]
    call = dict(n_offsets=4, num_heads_q=heads, num_heads_k=heads, total_q=sum(lengths), total_k=sum(lengths), max_seq_len_q=max_q,
                max_seq_len_k=max_k)  # fmt: skip
    size = sizes(**call)[0]
    blocks = (max_k + 31) // 32
    if max_q == max_k:
        assert size == heads * 128 * (((sum(lengths) + 32 * 3) * (blocks + 1) + 1) // 2)
    else:
        assert size == heads * 128 * sum(lengths) * (blocks | 1)
    # the sequences' first lines as the kernels place them, and the end of the last one
    first, ahead = sum(lengths[:-1]), 2
    rows = min(lengths[-1], max_q)
    end = (((first + 32 * ahead) * (blocks + 1) + 1) // 2 + pair_lines((rows + 31) // 32)) if max_q == max_k else (first + rows) * (blocks | 1)
    assert end <= size // heads // 128
