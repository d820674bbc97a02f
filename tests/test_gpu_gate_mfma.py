"""GPU parity of the 16-bit attention gate at dims that are a multiple of 64: groups of 16 and 32 tokens that
end anywhere, every head count and pack width of the fast path, every dim the matrix-core kernels are built
for, and more groups than blocks (several turns of the double-buffered backward, the last one partial).
Which of them run the matrix cores, each way, is decided by heads x dim and tokens; test_gpu_routes.py has
the cases on both sides."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_attention_gate import _check_ref_api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,heads,dh,dim", [
    (1, 8, 64, 512), (15, 2, 64, 64), (16, 4, 32, 128), (33, 4, 64, 192), (64, 8, 64, 256), (31, 16, 32, 384),
    (97, 8, 16, 512), (65, 2, 256, 192), (20001, 4, 32, 64), (33000, 8, 64, 128),
])
def test_gate_on_the_matrix_cores(hip_ext, dtype, m, heads, dh, dim):
    _check_ref_api(hip_ext, m, heads, dh, dim, dtype, 61)


def test_infinities_stay_in_their_token(hip_ext):
    """An infinite x row reaches its own gates and grad_W, not its neighbours' grad_x or gates."""
    m, h, dh, d = 40, 8, 64, 192
    g = torch.Generator().manual_seed(62)
    attn = torch.randn(m, h, dh, generator=g).to(torch.bfloat16).cuda()
    x = torch.randn(m, d, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(h, d, generator=g) / d**0.5).to(torch.bfloat16).cuda()
    b = torch.zeros(h, dtype=torch.bfloat16, device="cuda")
    gout = torch.randn(m, h * dh, generator=g).to(torch.bfloat16).cuda()
    x2 = x.clone()
    x2[39, 5] = float("inf")  # the last token: also what the tail of its group repeats
    o1, g1, *_ = hip_ext.attention_gate_forward(attn, x, w, b)
    o2, g2, *_ = hip_ext.attention_gate_forward(attn, x2, w, b)
    assert torch.equal(o1[:39], o2[:39]) and torch.equal(g1[:39], g2[:39])
    assert torch.equal(g2[39], (w[:, 5] > 0).to(torch.bfloat16))
    _, gx1, gw1, _ = hip_ext.attention_gate_backward(gout, attn, x, w, g1)
    _, gx2, gw2, _ = hip_ext.attention_gate_backward(gout, attn, x2, w, g1)
    assert torch.equal(gx1, gx2)
    keep = torch.ones(d, dtype=torch.bool)
    keep[5] = False
    assert torch.equal(gw1[:, keep], gw2[:, keep]) and torch.isinf(gw2[:, 5]).all()


def test_infinities_stay_in_their_token_at_many_products(hip_ext):
    """The same at heads x dim of 4096, where the forward runs the matrix cores at any number of tokens."""
    m, h, dh, d = 70, 8, 64, 512
    g = torch.Generator().manual_seed(64)
    attn = torch.randn(m, h, dh, generator=g).to(torch.bfloat16).cuda()
    x = torch.randn(m, d, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(h, d, generator=g) / d**0.5).to(torch.bfloat16).cuda()
    b = torch.zeros(h, dtype=torch.bfloat16, device="cuda")
    x2 = x.clone()
    x2[69, 5] = float("inf")
    o1, g1, *_ = hip_ext.attention_gate_forward(attn, x, w, b)
    o2, g2, *_ = hip_ext.attention_gate_forward(attn, x2, w, b)
    assert torch.equal(o1[:69], o2[:69]) and torch.equal(g1[:69], g2[:69])
    assert torch.equal(g2[69], (w[:, 5] > 0).to(torch.bfloat16))
