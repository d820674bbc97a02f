"""GPU parity: the grouped linear's backward products at more than 192 inputs and its tanh forward.

The backward cases are small grids, which the dispatch gives to the kernels with narrower blocks (all but
the dx of the case with 60 groups); the 256-wide tiles of grouped_gemm.hip are taken from the grid sizes
of test_gpu_routes.py, which holds the cases at their edges.  The tanh forward and the two-kernel mask MLP
run grouped_gemm.hip here."""

from __future__ import annotations

import pytest
import torch

import oracle
from tests.conftest import assert_parity, by_index, dt_name, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,groups,i,o", [
    (1, 3, 512, 32),       # one row, one K chunk
    (31, 2, 512, 64),      # dW below 32 rows: the register-staged kernel
    (32, 5, 384, 96),      # one dW K chunk
    (63, 2, 320, 160),     # dW chunk 0 with one row
    (257, 3, 264, 264),    # widths in whole eights, a tile of one row
    (150, 2, 768, 2048),   # a long K
    (513, 62, 192, 256),   # glin_dx and the DMA dW at 192 inputs
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tanh_of_every_pattern(hip_ext, dtype):
    """Zero weights leave z = the bias, so 32 groups of 2048 biases cover the 65536 patterns: every tanh
    equals the correctly rounded one of the table (NaN: any NaN)."""
    import ctypes

    import numpy as np

    from pymsst_amd._lib import dtype_code, load_library

    tab = np.zeros(1 << 15, dtype=np.uint16)
    assert load_library().pmsst_mask_mlp_tanh_table(dtype_code(dtype), tab.ctypes.data_as(ctypes.c_void_p), 1 << 15) == 0
    want = np.concatenate([tab, tab | 0x8000])
    want[0x8000] = 0  # the sum 0 w + (-0) is +0
    want = torch.from_numpy(want.view(np.int16)).cuda().view(dtype)
    bias = torch.arange(1 << 16, device="cuda").to(torch.int16).view(dtype).view(32, 2048)
    x = torch.zeros(3, 32, 32, dtype=dtype, device="cuda")
    w = torch.zeros(32, 2048, 32, dtype=dtype, device="cuda")
    got = hip_ext.grouped_linear_forward_act(x, w, bias, activation="tanh")
    for r in range(3):
        g = got[r].reshape(-1)
        assert torch.equal(torch.isnan(g), torch.isnan(want))
        assert torch.equal(g[~torch.isnan(g)].view(torch.int16), want[~torch.isnan(want)].view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,groups,i,o", [
    (1, 3, 32, 8),         # one row, one K chunk, one unit of outputs: the register-staged kernel
    (127, 2, 64, 256),     # two chunks
    (129, 5, 96, 384),     # a second row tile of one row; 192-wide output tiles
    (260, 3, 160, 264),    # five chunks, an output tile that ends after 72 of 192
    (300, 2, 512, 2048),
])
def test_wide_tanh_forward(hip_ext, dtype, m, groups, i, o):
    dn = dt_name(dtype)
    g = torch.Generator().manual_seed(53)
    x = torch.randn(m, groups, i, generator=g).to(dtype).cuda()
    w = (torch.randn(groups, o, i, generator=g) / i**0.5).to(dtype).cuda()
    b = (0.1 * torch.randn(groups, o, generator=g)).to(dtype).cuda()
    out = hip_ext.grouped_linear_forward_act(x, w, b, activation="tanh")
    assert_parity(out, oracle.grouped_linear_forward(to_np(x), to_np(w), to_np(b), dn, act="tanh"), dn, "tanh")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dims,dim", [((4, 8, 132, 200, 64), 384), ((260, 200, 196, 140), 64)])
def test_mask_mlp_two_kernels_equal_the_one_pass(hip_ext, dtype, dims, dim):
    """With the hidden layer stored these shapes run a hidden and a final kernel, without it the one
    pass: the same bits."""
    m, hidden, nb = 131, 160, len(dims)
    g = torch.Generator().manual_seed(54)
    x = torch.randn(m, nb, dim, generator=g).to(dtype).cuda()
    w1 = (torch.randn(nb, hidden, dim, generator=g) / dim**0.5).to(dtype).cuda()
    b1 = (0.1 * torch.randn(nb, hidden, generator=g)).to(dtype).cuda()
    w2 = torch.cat([(torch.randn(2 * d, hidden, generator=g) / hidden**0.5).reshape(-1) for d in dims]).to(dtype).cuda()
    b2 = (0.1 * torch.randn(2 * sum(dims), generator=g)).to(dtype).cuda()
    out, pre, hid = hip_ext.mask_mlp_forward(x, w1, b1, w2, b2, dims, save_hidden=True)
    out1, pre1, _ = hip_ext.mask_mlp_forward(x, w1, b1, w2, b2, dims, save_hidden=False)
    assert torch.equal(out, out1) and torch.equal(pre, pre1)
    assert_parity(hid, oracle.mask_mlp_hidden(to_np(x), to_np(w1), to_np(b1), dt_name(dtype)), dt_name(dtype), "hidden",
                  by_index(1))
