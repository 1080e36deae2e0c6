"""The forward kernel for short work lists at the head-dim slots 32 and 64 with an output that takes no 16-byte stores: the same bits, and nothing
beside the output is written."""

import pytest
import torch

import helpers
import ops_rec  # noqa: F401
from ops_rec import _ops, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GUARD = 256


@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("dim,dim_v", [(64, 64), (64, 16), (48, 48), (32, 32)])
def test_output_off_a_16_byte_boundary(dim, dim_v, bias, monkeypatch):
    helpers.set_switch(monkeypatch, "HSTU_MI355_SHORT", "1")
    w = workloads.make("rows", dtype=torch.bfloat16, device=DEV, seed=dim, batch=6, heads=2, dim=dim, dim_v=dim_v, lo=0, hi=0,
                       lengths=[1, 300, 128, 129, 0, 77], max_seq_len=300, rab_std=0.5 if bias else None)  # fmt: skip
    p = _ops.prepare_forward(w.q, w.k, w.v, None, w.attn_bias, 0, 300, 300, w.silu_scale, w.seq_offset, w.seq_offset, None, None, 0, w.alpha)
    assert p.kernel_name().endswith("_d64_rab_short" if bias else "_d64_short"), p.kernel_name()
    want = p.launch().clone()
    n = want.numel() * 2
    raw = torch.full((n + 2 * GUARD,), 0x5A, dtype=torch.uint8, device=DEV)
    assert raw.data_ptr() % 16 == 0
    p.params.out = raw.data_ptr() + GUARD + 8
    p.launch()
    torch.cuda.synchronize()
    assert torch.equal(raw[GUARD + 8 : GUARD + 8 + n].view(torch.bfloat16).view(want.shape), want)
    assert bool((raw[: GUARD + 8] == 0x5A).all()) and bool((raw[GUARD + 8 + n :] == 0x5A).all())
