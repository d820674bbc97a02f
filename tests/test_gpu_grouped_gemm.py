"""GPU parity: the grouped linear's backward products on the 256-wide tiles of grouped_gemm.hip, at the
edges of its tiles: one and several K chunks (the ring is 4 deep, the loop unrolled by two), rows and
widths that end inside a tile, a row count that is no multiple of 32 (dW's first K chunk is partial)."""

from __future__ import annotations

import pytest
import torch

import oracle
from tests.conftest import assert_parity, by_index, dt_name, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,groups,i,o", [
    (1, 3, 512, 32),       # one row, one K chunk
    (31, 2, 512, 64),      # dW below its 32 rows: the register-staged kernel
    (32, 5, 384, 96),      # one dW K chunk
    (63, 2, 320, 160),     # a second tile of 128 of its 192 columns; dW chunk 0 with one row
    (257, 3, 264, 264),    # a tile of 8 columns, a tile of one row; O no multiple of 32: dx elsewhere
    (150, 2, 768, 2048),   # three 256-wide tiles, 64 K chunks
    (513, 62, 192, 256),   # dW from 192 inputs on
    (129, 4, 256, 512),
])
def test_wide_grouped_backward(hip_ext, dtype, m, groups, i, o):
    dn = dt_name(dtype)
    g = torch.Generator().manual_seed(51)
    x = torch.randn(m, groups, i, generator=g).to(dtype).cuda()
    w = (torch.randn(groups, o, i, generator=g) / o**0.5).to(dtype).cuda()
    dy = torch.randn(m, groups, o, generator=g).to(dtype).cuda()
    for has_bias in (True, False):
        dx, dw, db = hip_ext.grouped_linear_backward(dy, x, w, has_bias)
        rdx, rdw, rdb = oracle.grouped_linear_backward(to_np(dy), to_np(x), to_np(w), has_bias, dn)
        assert_parity(dx, rdx, dn, "dx", by_index(1))
        assert_parity(dw, rdw, dn, "dW", by_index(0))
        if has_bias:
            assert_parity(db, rdb, dn, "db", by_index(0))


def test_wide_grouped_dx_where_the_rounds_fill(hip_ext):
    """192 inputs: 256-row blocks once whole rounds of one block per CU are 80 % full (here 60 x 11)."""
    m, groups, i, o, dtype = 2601, 60, 192, 96, torch.bfloat16
    g = torch.Generator().manual_seed(52)
    x = torch.randn(m, groups, i, generator=g).to(dtype).cuda()
    w = (torch.randn(groups, o, i, generator=g) / o**0.5).to(dtype).cuda()
    dy = torch.randn(m, groups, o, generator=g).to(dtype).cuda()
    dx, dw, db = hip_ext.grouped_linear_backward(dy, x, w, True)
    rdx, rdw, rdb = oracle.grouped_linear_backward(to_np(dy), to_np(x), to_np(w), True, "bf16")
    assert_parity(dx, rdx, "bf16", "dx", by_index(1))
    assert_parity(dw, rdw, "bf16", "dW", by_index(0))
    assert_parity(db, rdb, "bf16", "db", by_index(0))
