"""Which kernel a size runs, on both sides of the dispatch rules: the wide kernels stay off the sizes where
they measured slower than the kernels they replace (the figures stand at each rule)."""

from __future__ import annotations

import pytest
import torch

import oracle
from tests.conftest import assert_parity, by_index, dt_name, to_np

pytestmark = pytest.mark.gpu


def launched(call):
    """``(result, names)`` of the kernels that ``call`` launches."""
    from torch.profiler import ProfilerActivity, profile

    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA, ProfilerActivity.CPU]) as prof:
        out = call()
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert "_kernel" in names, "no kernel names recorded"
    return out, names


def _layer(m, groups, i, o, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(61)
    x = torch.randn(m, groups, i, generator=g).to(dtype).cuda()
    w = (torch.randn(groups, o, i, generator=g) / i**0.5).to(dtype).cuda()
    b = (0.1 * torch.randn(groups, o, generator=g)).to(dtype).cuda()
    return x, w, b, torch.randn(m, groups, o, generator=g).to(dtype).cuda()


@pytest.mark.parametrize("m,groups,i,o,wide", [
    (31, 62, 192, 64, False), (300, 5, 64, 120, False), (300, 5, 64, 128, True), (1, 1, 96, 264, True),
])
def test_tanh_forward(hip_ext, m, groups, i, o, wide):
    x, w, b, _ = _layer(m, groups, i, o)
    out, names = launched(lambda: hip_ext.grouped_linear_forward_act(x, w, b, activation="tanh"))
    assert ("gg_kernel" in names) == wide and ("bs_fwd_kernel" in names) != wide
    assert_parity(out, oracle.grouped_linear_forward(to_np(x), to_np(w), to_np(b), "bf16", act="tanh"), "bf16", "tanh")


def _check_backward(hip_ext, x, w, dy, dtype=torch.bfloat16):
    (dx, dw, db), names = launched(lambda: hip_ext.grouped_linear_backward(dy, x, w, True))
    dn = dt_name(dtype)
    rdx, rdw, rdb = oracle.grouped_linear_backward(to_np(dy), to_np(x), to_np(w), True, dn)
    assert_parity(dx, rdx, dn, "dx", by_index(1))
    assert_parity(dw, rdw, dn, "dW", by_index(0))
    assert_parity(db, rdb, dn, "db", by_index(0))
    return names


@pytest.mark.parametrize("m,groups,i,o,wide", [
    (1, 3, 512, 32, False), (90, 62, 512, 64, False), (91, 62, 512, 64, True),   # 2.75 blocks a CU from 90.8 rows
    (121, 62, 384, 64, False), (122, 62, 384, 96, True),                         # from 121.1 rows
    (1023, 8, 512, 64, False), (1024, 8, 512, 64, True),                         # 4 blocks a CU
    (129, 62, 320, 64, False), (146, 62, 320, 160, True), (173, 62, 264, 264, False),  # O no multiple of 32
])
def test_wide_input_gradient(hip_ext, m, groups, i, o, wide):
    x, w, _, dy = _layer(m, groups, i, o)
    names = _check_backward(hip_ext, x, w, dy)
    assert ("bs_bwd_dx_kernel" in names) != wide
