"""Which kernel a size runs, on both sides of the dispatch rules: the wide kernels stay off the sizes where
they measured slower than the kernels they replace (the figures stand at each rule)."""

from __future__ import annotations

import subprocess
import sys
from pathlib import Path

import numpy as np
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
    xd, dyd = (t.double().transpose(0, 1).contiguous() for t in (x, dy))
    assert_parity(dx, torch.matmul(dyd, w.double()).transpose(0, 1), dn, "dx", by_index(1))
    assert_parity(dw, torch.matmul(dyd.transpose(1, 2).contiguous(), xd), dn, "dW", by_index(0))
    assert_parity(db, dyd.sum(1), dn, "db", by_index(0))
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


@pytest.mark.parametrize("m,groups,i,o,wide", [
    (63, 62, 256, 768, False), (64, 62, 256, 768, True),       # 256-wide tiles, 6 rounds against one
    (97, 60, 256, 640, False),                                 # 5
    (128, 62, 384, 1536, False), (129, 62, 384, 1416, True),   # 192-wide, 6; an output tile that ends after 136
    (1399, 62, 192, 768, False), (1400, 62, 192, 768, True),   # 192-wide, 4.5
    (1500, 62, 192, 384, False),                               # 2.25
    (318, 62, 200, 800, True), (317, 62, 200, 800, False),     # no whole 64s: rows x 6.3 from 2000
    (800, 62, 200, 200, False), (700, 8, 200, 200, False),     # 3.9, 0.5
    (65, 2, 2048, 1024, True),                                 # few groups on few XCDs: 8
])
def test_wide_weight_gradient(hip_ext, m, groups, i, o, wide):
    x, w, _, dy = _layer(m, groups, i, o)
    names = _check_backward(hip_ext, x, w, dy)
    assert ("me_bwd_dw_dma_kernel" in names or "bs_bwd_dw_kernel" in names) != wide


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,groups,i,o", [
    (91, 62, 512, 32),      # dx: one K chunk
    (257, 62, 264, 1056),   # dx: a tile of one row, one of 8 columns; dW not wide
    (64, 62, 512, 1024),    # dW: two whole K chunks
    (65, 60, 768, 1032),    # dW: three 256-wide tiles, an output tile of 8, a first chunk of one row
    (161, 62, 384, 1536),   # dW: 192-wide tiles; dx: 48 K chunks
    (416, 62, 264, 1056),   # both at a width in whole eights only
])
def test_wide_tiles_at_their_edges(hip_ext, dtype, m, groups, i, o):
    x, w, _, dy = _layer(m, groups, i, o, dtype)
    assert "gg_kernel" in _check_backward(hip_ext, x, w, dy, dtype)


@pytest.mark.parametrize("m,dim,dims,two", [
    (256, 192, (260, 200, 196, 140), False), (257, 192, (260, 200, 196, 140), True),
    (256, 128, (260, 200, 196, 140), False), (257, 128, (260, 200, 196, 140), True),
    (768, 64, (260, 200, 196, 140), False), (769, 64, (260, 200, 196, 140), True),
    (3, 256, (260, 200, 196, 140), True), (3, 256, (8, 64, 132), False), (3, 384, (8, 64, 132), True),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mask_mlp_forward(hip_ext, dtype, m, dim, dims, two):
    """Both forms give the same bits: the call without the stored hidden layer always runs the one pass."""
    hidden, nb = 160, len(dims)
    g = torch.Generator().manual_seed(62)
    x = torch.randn(m, nb, dim, generator=g).to(dtype).cuda()
    w1 = (torch.randn(nb, hidden, dim, generator=g) / dim**0.5).to(dtype).cuda()
    b1 = (0.1 * torch.randn(nb, hidden, generator=g)).to(dtype).cuda()
    w2 = torch.cat([(torch.randn(2 * d, hidden, generator=g) / hidden**0.5).reshape(-1) for d in dims]).to(dtype).cuda()
    b2 = (0.1 * torch.randn(2 * sum(dims), generator=g)).to(dtype).cuda()
    (out, pre, hid), names = launched(lambda: hip_ext.mask_mlp_forward(x, w1, b1, w2, b2, dims, save_hidden=True))
    assert ("gg_kernel" in names) == two and ("mlp_fwd_kernel" in names) != two
    out1, pre1, _ = hip_ext.mask_mlp_forward(x, w1, b1, w2, b2, dims)
    assert torch.equal(out, out1) and torch.equal(pre, pre1)
    assert_parity(hid, oracle.mask_mlp_hidden(to_np(x), to_np(w1), to_np(b1), dt_name(dtype)), dt_name(dtype), "hidden",
                  by_index(1))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,heads,dh,dim,fwd,bwd", [
    (1, 8, 64, 512, True, True), (33, 16, 32, 256, True, True), (31, 16, 16, 384, True, False),  # 16 x 384: generic
    (47, 8, 64, 384, False, True), (8193, 8, 64, 256, True, True), (8191, 8, 64, 256, False, True),
    (8192, 4, 32, 192, False, False), (16384, 4, 32, 192, True, False), (1999, 8, 16, 128, False, False),
    (2000, 8, 16, 128, False, True), (15, 8, 64, 192, False, True), (65, 16, 16, 128, False, True),
    (16421, 2, 64, 64, True, False), (3001, 16, 8, 64, False, True), (16400, 4, 64, 128, True, False),
])
def test_attention_gate(hip_ext, dtype, m, heads, dh, dim, fwd, bwd):
    """The matrix-core gate on both sides of its rules, at groups of 64 and 32 tokens that end anywhere and at
    each dim it is built for."""
    dn = dt_name(dtype)
    g = torch.Generator().manual_seed(63)
    attn = torch.randn(m, heads, dh, generator=g).to(dtype).cuda()
    x = torch.randn(m, dim, generator=g).to(dtype).cuda()
    w = (torch.randn(heads, dim, generator=g) / dim**0.5).to(dtype).cuda()
    b = (0.1 * torch.randn(heads, generator=g)).to(dtype).cuda()
    gout = torch.randn(m, heads * dh, generator=g).to(dtype).cuda()
    (out, gate, *_), names = launched(lambda: hip_ext.attention_gate_forward(attn, x, w, b))
    assert ("gate_mfma_fwd_kernel" in names) == fwd
    r_out, r_gate = oracle.attention_gate_forward(to_np(attn), to_np(x), to_np(w), to_np(b), dn)[:2]
    assert_parity(out, r_out.reshape(m, -1), dn, "out")
    assert_parity(gate, r_gate, dn, "gate")
    (ga, gx, gw, gb), names = launched(lambda: hip_ext.attention_gate_backward(gout, attn, x, w, gate))
    assert ("gate_mfma_bwd_kernel" in names) == bwd
    refs = oracle.attention_gate_backward(to_np(gout), to_np(attn), to_np(x), to_np(w), to_np(gate), dn)
    for got, want, what in zip((ga, gx, gw, gb), refs, ("grad_attn", "grad_x", "grad_W", "grad_b")):
        assert_parity(got, np.asarray(want).reshape(got.shape), dn, what)


_CAPTURE_AFTER_WARM_UP = """
import torch
from pymsst_amd.fused_extension import load_fused_band_split_extension
ext = load_fused_band_split_extension()
dims, dim, hidden, m = (8, 64, 132), 384, 160, 70
g = torch.Generator().manual_seed(64)
x = torch.randn(m, len(dims), dim, generator=g).bfloat16().cuda()
w1 = (torch.randn(len(dims), hidden, dim, generator=g) / dim**0.5).bfloat16().cuda()
b1 = torch.randn(len(dims), hidden, generator=g).bfloat16().cuda()
w2 = (torch.randn(2 * sum(dims) * hidden, generator=g) / hidden**0.5).bfloat16().cuda()
b2 = torch.randn(2 * sum(dims), generator=g).bfloat16().cuda()
want = ext.mask_mlp_forward(x, w1, b1, w2, b2, dims, save_hidden=True)
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    got = ext.mask_mlp_forward(x, w1, b1, w2, b2, dims)
for _ in range(3):
    got[0].zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
print("captured")
"""


def test_capture_of_the_one_pass_after_a_two_kernel_warm_up(hip_ext):
    """A process of its own: the device's tanh tables are uploaded once."""
    run = subprocess.run([sys.executable, "-c", _CAPTURE_AFTER_WARM_UP], cwd=Path(__file__).resolve().parents[1],
                         capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and "captured" in run.stdout, run.stderr[-2000:]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [384, 512])
def test_one_pass_with_the_hidden_layer_at_wide_dims(hip_ext, dtype, dim):
    """A first bias that is not 8-byte aligned keeps dims 384 and 512 on the one pass, with the hidden layer
    stored and with the mask product: the bits of the aligned call."""
    dims, hidden, batch, frames, stems, channels = (8, 64, 132), 160, 2, 35, 2, 2
    m, nb, total = batch * frames, len(dims), sum(dims)
    g = torch.Generator().manual_seed(65)
    x = torch.randn(m, nb, dim, generator=g).to(dtype).cuda()
    w1 = (torch.randn(nb, hidden, dim, generator=g) / dim**0.5).to(dtype).cuda()
    b1 = (0.1 * torch.randn(nb * hidden + 1, generator=g)).to(dtype).cuda()[1:].view(nb, hidden)
    w2 = (torch.randn(2 * total * hidden, generator=g) / hidden**0.5).to(dtype).cuda()
    b2 = (0.1 * torch.randn(2 * total, generator=g)).to(dtype).cuda()
    spec = torch.view_as_complex(torch.randn(batch, total // 2, frames, 2, generator=g)).cuda()

    def apply(bias):
        est = torch.zeros(batch * stems * channels, total // 2 // channels, frames, dtype=torch.complex64, device="cuda")
        pre, hid = hip_ext.mask_mlp_forward_apply(x, w1, bias, w2, b2, dims, spec, est, 1, channels, save_hidden=True)
        return pre, hid, torch.view_as_real(est)

    for call in (lambda b: hip_ext.mask_mlp_forward(x, w1, b, w2, b2, dims, save_hidden=True), apply):
        one, names = launched(lambda: call(b1))
        assert "mlp_fwd_kernel" in names and "gg_kernel" not in names
        two, names = launched(lambda: call(b1.clone()))
        assert "gg_kernel" in names
        assert all(torch.equal(a, b) for a, b in zip(one, two))
