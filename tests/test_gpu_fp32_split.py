"""fp32 products (gemm.h): as exact as the fp32 sums, also for what three bf16 parts cannot hold.

Most of these sizes are below gemm.h's rule for the split into bf16 parts and run the fp32 matrix
instructions, whose results the split has to match; test_gpu_fp32_routes.py asks the same of sizes that
are split.

* Error against 64 bits, at the sizes where the K loop can go wrong (one partial chunk, several), no
  larger than sqrt(K) / 2 rounding errors of the fp32 sum: 2^-24 (1 + sqrt(K) / 2) of the result's RMS
  times sqrt(2), measured 0.8 of it (0.3 split).
* Exponents from -60 to 60 (test_gpu_fp32_routes.py: from 2^-124).
* An infinity, a NaN, a value above bf16's largest, an overflow: the results of a plain fp32 product.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(m, groups, i, o, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, groups, i, generator=g).cuda()
    w = (torch.randn(groups, o, i, generator=g) / i**0.5).cuda()
    return x, w, torch.randn(m, groups, o, generator=g).cuda()


def _exact(x, w, dy):
    x, w, dy = x.double(), w.double(), dy.double()
    return (torch.stack([x[:, b] @ w[b].t() for b in range(w.shape[0])], 1),
            torch.stack([dy[:, b] @ w[b] for b in range(w.shape[0])], 1),
            torch.stack([dy[:, b].t() @ x[:, b] for b in range(w.shape[0])], 0))


@pytest.mark.parametrize("m,groups,i,o", [(1, 1, 1, 1), (33, 3, 7, 10), (65, 2, 32, 64), (130, 5, 64, 256),
                                          (257, 3, 100, 132), (1032, 2, 192, 768)])
def test_error_is_that_of_fp32_sums(hip_ext, m, groups, i, o):
    x, w, dy = _case(m, groups, i, o)
    out = hip_ext.grouped_linear_forward(x, w)
    dx, dw, _ = hip_ext.grouped_linear_backward(dy, x, w, False)
    for got, want, k in zip((out, dx, dw), _exact(x, w, dy), (i, o, m)):
        rel = ((got.double() - want).norm() / want.norm()).item()
        assert rel <= 2.0**-23.5 * (1 + k**0.5 / 2), (rel, k)


@pytest.mark.parametrize("exp", [-60, -20, 20, 60])
def test_any_exponent(hip_ext, exp):
    x, w, dy = _case(70, 2, 96, 64, seed=1)
    base = hip_ext.grouped_linear_forward(x, w)
    assert torch.equal(hip_ext.grouped_linear_forward(x * 2.0**exp, w), base * 2.0**exp)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_values_bf16_cannot_hold(hip_ext, bad):
    """Row 5 of x holds the value: its outputs are those of an fp32 product (3.4e38 rounds to infinity in
    bf16), every other row's are those without it."""
    x, w, dy = _case(130, 2, 64, 96, seed=2)
    clean = hip_ext.grouped_linear_forward(x, w)
    x2 = x.clone()
    x2[5, 1] = 0.0
    x2[5, 1, 7] = bad
    out = hip_ext.grouped_linear_forward(x2, w)
    want = bad * w[1, :, 7]
    assert torch.equal(torch.isnan(out[5, 1]), torch.isnan(want))
    fine = ~torch.isnan(want)
    assert torch.equal(out[5, 1][fine], want[fine])
    keep = torch.ones(130, dtype=torch.bool)
    keep[5] = False
    assert torch.equal(out[:, 0], clean[:, 0])
    assert torch.allclose(out[keep][:, 1], clean[keep][:, 1], rtol=1e-5, atol=1e-5)


def test_norm_and_bias_sums_after_a_rerun(hip_ext):
    """The band split's row norms and the bias column sums are gathered by the K loop: a block that runs
    it twice (an infinity in dy) still counts every row once."""
    x, w, dy = _case(130, 2, 64, 96, seed=3)
    _, _, db = hip_ext.grouped_linear_backward(dy, x, w, True)
    dy2 = dy.clone()
    dy2[3, 0, 11] = float("inf")
    _, _, db2 = hip_ext.grouped_linear_backward(dy2, x, w, True)
    assert db2[0, 11] == float("inf")
    keep = torch.ones(96, dtype=torch.bool)
    keep[11] = False
    assert torch.equal(db2[0][keep], db[0][keep]) and torch.equal(db2[1], db[1])
