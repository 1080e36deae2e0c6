"""A workspace smaller than the forward asks for, at the head-dim slot whose work list cuts no items: the call runs as far as the room goes."""

import pytest
import torch

import helpers
from ops_rec import _ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("parts", [0, 1, 2, 3, 31, 32, 33, 255, 256])
def test_room_for_few_partial_outputs_at_the_slot_256(parts, monkeypatch):
    """16 items at a slot whose list splits nothing: they are cut into two parts and more from room for 32 on, and up to there run as they do
    without room, where the rows have the bits of whole items (the last bit of a row may differ between both: rtol 2^-7)."""
    rows, keys = [80, 77, 1, 64], [4096, 4000, 2500, 3001]
    g = torch.Generator().manual_seed(5)
    q = (torch.randn(sum(rows), 4, 256, generator=g) * 0.5).to(torch.bfloat16).to(DEV)
    k, v = ((torch.randn(sum(keys), 4, 256, generator=g) * 0.5).to(torch.bfloat16).to(DEV) for _ in range(2))
    offs, offs_k = (torch.tensor([0] + n, dtype=torch.int32).cumsum(0).to(torch.int32).to(DEV) for n in (rows, keys))

    def call():
        return _ops.prepare_forward(q, k, v, None, None, 0, max(rows), max(keys), 1.0 / 4096, offs, offs_k, None, None, 0, 1.0 / 16)

    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", "0")
    whole = call().launch().clone()
    helpers.set_switch(monkeypatch, "HSTU_MI355_SPLIT", None)
    p = call()
    assert p.kernel_name().endswith("_split") and p.workspace_bytes == 16384 + 256 * 128 * 256 * 4
    p.workspace_bytes = 16384 + parts * 128 * 256 * 4 if parts else 0
    p.workspace = torch.full((p.workspace_bytes,), 0x5A, dtype=torch.uint8, device=DEV) if parts else None
    p.out.fill_(float("nan"))
    out = p.launch()
    if parts < 32:
        assert torch.equal(out, whole)
    else:
        torch.testing.assert_close(out.float(), whole.float(), atol=2e-7, rtol=2**-7)
