"""in_linear_silu: which calls take the kernel with the weights in registers, both sides of each line of the rule (on 256 compute units, what the
library assumes where there is no device; nothing is launched)."""

import ctypes

import pytest

from ops_rec import _native


@pytest.mark.parametrize(
    "m,n,k,rows",
    [
        (20480, 2048, 512, True),
        (6143, 2048, 512, False),  # 32 groups of rows: six tiles are 6144
        (6144, 2048, 512, True),
        (1920, 6144, 384, True),  # 24 column blocks, 10 groups
        (1919, 6144, 384, False),
        (5119, 7680, 384, False),  # 30 blocks, 8 groups: 20 tiles are 5120
        (5120, 7680, 384, True),
        (1279, 22528, 512, False),  # 88 blocks, two groups, 80 compute units idle
        (1280, 22528, 512, True),
        (5119, 8192, 512, False),  # 32 blocks, 8 groups: no compute unit idle, but few blocks
        (768, 16384, 512, True),  # 64 blocks
        (767, 16384, 512, False),
        (1152, 10304, 368, True),  # k = 11.5 steps of the other kernel
        (1151, 10304, 368, False),
        (25600, 1920, 160, False),
        (8191, 1920, 160, True),  # 32 groups: less than eight tiles
        (8192, 1920, 160, False),
        (6143, 1920, 160, False),
        (30462, 1408, 176, True),
        (50000, 2560, 128, False),
        (50000, 2112, 528, False),
    ],
    ids=str,
)
def test_the_rule(m, n, k, rows):
    p = _native.new_in_linear_silu_params()
    p.x, p.weight, p.bias = 0x1000, 0x2000, 0x3000  # never dereferenced
    p.user, p.value, p.query, p.key, p.linear_output = 0x4000, 0x5000, 0x6000, 0x7000, 0x8000
    p.m, p.n, p.k, p.dtype = m, n, k, _native.DT_BF16
    parts = [n // 256] * 3
    for i, part in enumerate(parts + [n // 64 - sum(parts)]):
        p.split[i] = 64 * part
    name = _native.load().in_linear_silu_fwd_kernel_name(ctypes.byref(p))
    assert name is not None, _native.last_error()
    assert ("_rows" in name.decode()) == rows, name
