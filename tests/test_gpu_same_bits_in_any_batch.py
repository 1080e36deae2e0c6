"""HSTU_MI355_SPLIT=0, at head dims above 64 with HSTU_MI355_SHORT=0 beside it: the rows of a sequence of more than 64 rows are the same bits
whatever else is in the batch.  HSTU_MI355_SHORT=1 still forces the kernel for short lists."""

import pytest
import torch

import helpers
from ops_rec import _ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("dim,short", [(32, None), (48, None), (64, None), (128, "0"), (192, "0")])
def test_with_splitting_off(dim, short, bias, monkeypatch):
    gen = torch.Generator().manual_seed(dim)
    first = [(torch.randn(200, 2, dim, generator=gen) * 0.7).to(torch.bfloat16) for _ in range(3)]
    first_bias = (torch.randn(2, 200, 200, generator=gen) * 0.3).to(torch.bfloat16)

    def call(more):  # the rows of the first sequence, and the kernel that the batch takes
        lengths = [200] + more
        n = -(-max(lengths) // 8) * 8
        q, k, v = (torch.cat((t, (torch.randn(sum(more), 2, dim, generator=gen) * 0.7).to(torch.bfloat16))).to(DEV) for t in first)
        rab = None
        if bias:
            rab = torch.zeros(len(lengths), 2, n, n, dtype=torch.bfloat16, device=DEV)
            rab[0, :, :200, :200] = first_bias.to(DEV)
        offs = torch.tensor([0] + lengths).cumsum(0).to(torch.int32).to(DEV)
        p = _ops.prepare_forward(q, k, v, None, rab, 0, n, n, 1 / 256, offs, offs, None, None, 0, dim**-0.5)
        return p.launch()[:200].clone(), p.kernel_name()

    batches = ([], [100], [1100], [150] * (800 if bias else 2000))
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", short)
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    rows, names = zip(*map(call, batches))
    assert not any(name.endswith(("_short", "_split")) for name in names) and len(set(names)) > 1, names
    for other in rows[1:]:
        assert torch.equal(other, rows[0])
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "1")
    assert call([])[1].endswith("_short") == (dim <= 128)
