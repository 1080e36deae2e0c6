"""Long lists at the head-dim slots 32 and 64: which calls leave the kernel for short work lists to the queues because heads share lines of K and
V, both sides of each line of the rule on 256 compute units, and the queues' result against the CPU oracle."""

import pytest
import torch

import ops_rec  # noqa: F401
from ops_rec import _ops, workloads
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize(
    "batch,heads,heads_k,dim,dim_v,rows,short",
    [
        (256, 4, 4, 48, 48, 257, False),  # 3072 slots
        (255, 4, 4, 48, 48, 257, True),
        (512, 4, 4, 48, 48, 256, True),
        (256, 4, 4, 64, 48, 257, False),
        (256, 4, 4, 48, 16, 257, False),
        (256, 4, 4, 64, 64, 257, True),  # whole lines
        (256, 4, 4, 64, 32, 257, True),  # halves of lines
        (256, 4, 2, 48, 48, 257, True),  # grouped heads
        (1024, 1, 1, 48, 48, 257, True),  # one head: rows side by side
        (1451, 4, 4, 32, 32, 257, False),  # 17412 slots
        (1450, 4, 4, 32, 32, 257, True),
        (1451, 4, 2, 32, 16, 257, False),
        (2048, 8, 8, 16, 16, 256, True),
    ],
    ids=str,
)
def test_the_rule(batch, heads, heads_k, dim, dim_v, rows, short):
    q = torch.empty(batch * rows, heads, dim, dtype=torch.bfloat16, device=DEV)
    k = torch.empty(batch * rows, heads_k, dim, dtype=torch.bfloat16, device=DEV)
    v = torch.empty(batch * rows, heads_k, dim_v, dtype=torch.bfloat16, device=DEV)
    offs = (torch.arange(batch + 1, dtype=torch.int32) * rows).to(DEV)
    p = _ops.prepare_forward(q, k, v, None, None, 0, rows, rows, 1.0 / rows, offs, offs, None, None, 0, 0.125)
    assert p.kernel_name().endswith("_short" if short else "_queues"), p.kernel_name()


def test_result():
    lengths = [400, 257, 1, 129] * 65
    w = workloads.make("long", batch=len(lengths), heads=4, dim=48, dim_v=48, lo=0, hi=0, lengths=lengths, dtype=torch.bfloat16, std=0.5, seed=48)
    d = w.to(DEV)
    p = _ops.prepare_forward(d.q, d.k, d.v, None, None, 0, d.max_seq_len, d.max_seq_len, d.silu_scale, d.seq_offset, d.seq_offset, None, None, 0, d.alpha)
    assert p.kernel_name().endswith("_queues"), p.kernel_name()
    ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
    torch.testing.assert_close(p.launch().float().cpu(), ref, atol=1e-2, rtol=1e-2)
