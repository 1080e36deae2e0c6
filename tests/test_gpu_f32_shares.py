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


@pytest.mark.parametrize("dim", [32, 64, 128, 256])
def test_without_shares_a_sequence_has_the_same_bits_in_any_batch(dim, monkeypatch):
    lengths = [333, 20, 700, 1]
    w = workloads.make("f32", batch=4, heads=2, dim=dim, lo=0, hi=0, lengths=lengths, max_seq_len=700, dtype=torch.float32, std=0.5,
                       seed=dim, device=DEV)  # fmt: skip
    attend = lambda q, k, v, offs: ops_rec.ascendc.attention.hstu_jagged(q, k, v, None, None, 0, 700, 1.0, offs, None, None, 0, w.alpha)  # noqa: E731

    def alone_and_together():
        one = attend(*(t[:333].contiguous() for t in (w.q, w.k, w.v)), w.seq_offset[:2].contiguous())
        many = [t.repeat(100, 1, 1) for t in (w.q, w.k, w.v)]
        offs = torch.cat([w.seq_offset[:-1] + i * w.seq_offset[-1] for i in range(100)] + [100 * w.seq_offset[-1:]])
        return one, attend(*many, offs)[:333]

    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    one, together = alone_and_together()
    assert torch.equal(one, together)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", None)
    one, together = alone_and_together()  # (the documented default: to rounding)
    torch.testing.assert_close(one, together, atol=1e-5 * float(one.abs().max()), rtol=1e-5)
