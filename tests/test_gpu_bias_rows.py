"""attn_bias rows that start anywhere: max_seq_len of every residue modulo 4 and tensors that start in the middle of a 4-byte word.

The persistent forward kernel reads the aligned words that hold a lane's values and shifts them into place; the values that reach the products
are the same whatever the pitch, so the outputs are compared bit for bit with the same values in rows of a multiple of 8, and with the
CPU oracle.
"""

import pytest
import torch

import helpers
import ops_rec  # noqa: F401
from ops_rec import _ops, workloads
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LISTS = {
    "direct": dict(lengths=[1, 37, 130, 33, 0, 128]),
    "plain": dict(lengths=[300, 129, 700, 31, 257, 1] * 12),
    "long sweeps": dict(lengths=[900, 33, 1500], num_context=3, max_target=20, target_group_size=2, heads_k=1),
}


@pytest.mark.parametrize("start", [0, 1])
@pytest.mark.parametrize("more", [0, 1, 2, 3])
@pytest.mark.parametrize("dim,dtype", [(32, torch.bfloat16), (64, torch.float16), (128, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("name", list(LISTS))
def test_rows_that_start_anywhere(name, dim, dtype, more, start, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "0")  # (kernels of their own take some of the aligned ones)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    kw = LISTS[name]
    longest = (max(kw["lengths"]) + 3) // 4 * 4 + more
    w = workloads.make(name, batch=len(kw["lengths"]), heads=2, dim=dim, lo=0, hi=0, dtype=dtype, std=0.5, seed=dim + more, device=DEV,
                       max_seq_len=longest, **kw)  # fmt: skip
    n, wide = longest, (longest + 7) // 8 * 8
    g = torch.Generator(device=DEV).manual_seed(more)
    values = torch.randn(len(kw["lengths"]), 2, n, n, generator=g, device=DEV).mul_(0.5).to(dtype)
    flat = torch.full((values.numel() + 3,), float("nan"), dtype=dtype, device=DEV)  # (neighbours that must not be used)
    bias = flat[start : start + values.numel()].view_as(values)
    bias.copy_(values)
    padded = torch.zeros(values.shape[0], 2, wide, wide, dtype=dtype, device=DEV)
    padded[:, :, :n, :n] = values

    def run(b):
        p = _ops.prepare_forward(w.q, w.k, w.v, None, b, 0, b.shape[3], b.shape[3], 1.0 / n, w.seq_offset, w.seq_offset, w.num_context,
                                 w.num_target, w.target_group_size, w.alpha)  # fmt: skip
        return p.launch()

    out = run(bias)
    assert torch.equal(out, run(padded))
    if dim == 128 and name == "direct":
        c = w.to("cpu")
        ref = O.hstu_jagged_forward(c.q, c.k, c.v, out_dtype=torch.float32, **dict(c.oracle_kwargs(), attn_bias=values.cpu(), silu_scale=1.0 / n))
        torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
