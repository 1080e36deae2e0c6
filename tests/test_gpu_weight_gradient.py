"""in_linear_silu_bwd_weight of the C ABI (element-wise stage, weight gradient and column sums) against the element-wise kernel and
a float64 product of what it wrote: rows at the edges of the 32-row steps and of the chunks, columns of d_mixed at the edges
of the 128-column tiles with gradients that meet inside one, every tile width of x and its edges."""

import pytest
import torch

from ops_rec import _activation

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,split,k", [
    (1, [16, 16, 16, 16], 16), (31, [16, 64, 32, 80], 48), (33, [128, 128, 128, 128], 128), (300, [48, 48, 80, 144], 144),
    (4100, [64, 64, 64, 64], 64), (257, [256, 256, 256, 256], 256), (640, [16, 240, 64, 192], 272), (2085, [512] * 4, 512),
    (96, [544, 512, 528, 528], 528), (513, [1024] * 4, 1024), (20000, [32, 32, 32, 32], 16),
])  # fmt: skip
def test_against_the_stage_and_a_double_product(m, split, k, dtype):
    g = torch.Generator(device=DEV).manual_seed(m + k)
    n = sum(split)
    lin = torch.randn(m, n, generator=g, device=DEV).to(dtype)
    grads = [torch.randn(m, s, generator=g, device=DEV).to(dtype) for s in split]
    x = torch.randn(m, k, generator=g, device=DEV).to(dtype)
    d_mixed, weight_grad, sums = _activation.silu_backward_with_weight(lin, grads, split, x)
    want_d, want_sums = _activation.silu_backward_stage(lin, grads, split)
    assert torch.equal(d_mixed, want_d)
    torch.testing.assert_close(sums, want_sums, atol=1e-4 * m**0.5, rtol=1e-4)
    want = want_d.double().t() @ x.double()
    assert (weight_grad.double() - want).norm() <= 3e-3 * want.norm()
    again = _activation.silu_backward_with_weight(lin, grads, split, x, want_bias_grad=False)
    assert again[2] is None and torch.equal(again[1], weight_grad) and torch.equal(again[0], d_mixed)


@pytest.mark.parametrize("m,n,k", [(20000, 1024, 16), (20000, 8192, 1024), (30001, 8192, 512), (4096, 16384, 1024)])
def test_column_sums_are_as_close_to_64_bits_as_the_stage_alone(m, n, k):
    """A chunk of a wide weight is thousands of rows long: its sums are taken in two levels, as close to the 64-bit sums as those of the
    element-wise kernel, which adds blocks of 64 rows (within a quarter: the two round at other places)."""
    g = torch.Generator(device=DEV).manual_seed(m + k)
    split = [n // 4] * 4
    lin = torch.randn(m, n, generator=g, device=DEV).bfloat16()
    grads = [torch.randn(m, n // 4, generator=g, device=DEV).bfloat16() for _ in split]
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    sums, stage = _activation.silu_backward_with_weight(lin, grads, split, x)[2], _activation.silu_backward_stage(lin, grads, split)[1]
    z, s = lin.double(), torch.sigmoid(lin.double())
    want = (torch.cat(grads, 1).double() * s * (1 + z * (1 - s))).sum(0)
    assert (sums.double() - want).norm() <= 1.25 * (stage.double() - want).norm()
