"""The arrival counters of split items are told apart by the number of their launch, not cleared ahead of it: a workspace may hold
anything, a launch may follow another in the same workspace at once, a replayed launch repeats its number; and a workspace with
room for fewer partial outputs than the split would use splits as far as the room goes."""

import pytest
import torch

from ops_rec import _ops, workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def prepared(lengths, dim):
    w = workloads.make("split", batch=len(lengths), heads=2, dim=dim, lo=0, hi=0, lengths=lengths, seed=dim, device=DEV)
    return _ops.prepare_forward(w.q, w.k, w.v, None, None, 0, w.max_seq_len, w.max_seq_len, w.silu_scale, w.seq_offset,
                                w.seq_offset, None, None, 0, w.alpha)  # fmt: skip


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lengths", [[3000], [700, 2049, 1500], [130] * 7 + [5000]], ids=str)
def test_whatever_the_workspace_holds(lengths, dim):
    p = prepared(lengths, dim)
    assert p.kernel_name().endswith("_split")
    want = p.launch().clone()
    g = torch.Generator(device=DEV).manual_seed(0)
    for fill in (lambda ws: ws.fill_(0xFF), lambda ws: ws.zero_(), lambda ws: ws.random_(0, 256, generator=g), lambda ws: None):
        fill(p.workspace)
        for _ in range(3):
            p.out.fill_(float("nan"))
            assert torch.equal(p.launch(), want)


@pytest.mark.parametrize("parts", [2, 3, 17])
def test_room_for_few_partial_outputs(parts):
    p = prepared([4000, 900], 128)
    want = p.launch().clone()
    p.workspace_bytes = 16384 + parts * 128 * 128 * 4
    p.workspace = torch.full((p.workspace_bytes,), 0x5A, dtype=torch.uint8, device=DEV)
    p.out.fill_(float("nan"))
    got = p.launch()
    torch.testing.assert_close(got.float(), want.float(), atol=1e-2, rtol=1e-2)  # (other sums: rounding)


def test_replays_of_one_launch():
    p = prepared([2500, 64], 128)
    want = p.launch().clone()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        p.launch()
    for i in range(4):
        p.out.fill_(float("nan"))
        if i % 2:
            p.workspace.random_(0, 256)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(p.out, want)
