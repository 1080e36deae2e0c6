"""The fp32 forward kernel with a row group's keys dealt over 1 .. 8 wavefronts, against the CPU oracle: row counts at the edges of
its 16-row groups, key counts at the edges of its 16-key blocks and below one block per share, every head-dim slot."""

import pytest
import torch

import helpers
import ops_rec
from oracle import hstu_oracle as O
from ops_rec import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("split", ["0", None], ids=["one share", "shares"])
@pytest.mark.parametrize("dim,dim_v", [(32, 32), (24, 16), (64, 48), (128, 128), (200, 256)])
@pytest.mark.parametrize("lengths", [[1], [15, 16, 17], [127, 128, 129, 130, 0, 33], [1025, 31]], ids=str)
def test_against_the_oracle(lengths, dim, dim_v, split, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", split)
    for kw in (dict(), dict(rab_std=0.3, num_context=2, max_target=5, target_group_size=2)):
        w = workloads.make("f32", batch=len(lengths), heads=2, heads_k=1, dim=dim, dim_v=dim_v, lo=0, hi=0, lengths=lengths,
                           dtype=torch.float32, std=0.5, seed=len(lengths) + dim, **kw)  # fmt: skip
        out = ops_rec.ascendc.attention.hstu_jagged(*w.to(DEV).op_args())
        ref = O.hstu_jagged_forward(w.q, w.k, w.v, out_dtype=torch.float32, **w.oracle_kwargs())
        torch.testing.assert_close(out.cpu(), ref, atol=1e-5, rtol=1e-4)
