"""fp32 products on both sides of the rule that splits large ones into bf16 parts (gemm.h).

Below it a result is the chain of fused multiply-adds over k that the fp32 matrix cores compute, bit for
bit: the tiny model's steps, whose L1 loss turns a change of 1e-7 in its estimate into one of 2e-3 in its
gradients when an element passes its target, keep their outputs.  The chain is emulated in 64-bit
significands (a product of two fp32 numbers is exact in 48 bits; rounding the sum to 64 bits first changes
the fp32 result with a chance of 2^-40 an element).  Above it the error against 64 bits stays below
sqrt(K) / 2 roundings of the fp32 sum, also for numbers that three bf16 parts cannot hold.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_parity, by_band, by_index, to_np
from tests.test_gpu_band_split import BSR_WIDTHS, _check_ragged

pytestmark = pytest.mark.gpu


def _chain(a, b):
    """``sum_k a[m, k] b[n, k]``, one fp32 rounding a term, in order of k."""
    a, b = a.cpu().numpy().astype(np.longdouble), b.cpu().numpy().astype(np.longdouble)
    acc = np.zeros((a.shape[0], b.shape[0]), np.float32)
    for k in range(a.shape[1]):
        acc = (acc + a[:, k, None] * b[None, :, k]).astype(np.float32)
    return torch.from_numpy(acc)


def _layer(m, groups, i, o, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, groups, i, generator=g)
    w = torch.randn(groups, o, i, generator=g) / i**0.5
    return x, w, torch.randn(m, groups, o, generator=g)


@pytest.mark.parametrize("m,groups,i,o", [(1, 1, 1, 1), (33, 3, 7, 10), (65, 2, 36, 64), (130, 62, 64, 256),
                                          (97, 62, 192, 256)])  # the last: 0.295 G multiply-adds, just below the rule
def test_small_products_are_fused_chains(hip_ext, m, groups, i, o):
    x, w, dy = _layer(m, groups, i, o, 5)
    out = hip_ext.grouped_linear_forward(x.cuda(), w.cuda()).cpu()
    dx, dw, _ = hip_ext.grouped_linear_backward(dy.cuda(), x.cuda(), w.cuda(), False)
    for g in {0, groups - 1}:
        assert torch.equal(out[:, g], _chain(x[:, g], w[g]))
        assert torch.equal(dx[:, g].cpu(), _chain(dy[:, g], w[g].t()))
        assert torch.equal(dw[g].cpu(), _chain(dy[:, g].t(), x[:, g].t()))


def test_the_tiny_models_final_layer_is_a_fused_chain(hip_ext):
    m, h = 130, 256  # 0.273 G multiply-adds, the tiny step's largest launch
    g = torch.Generator().manual_seed(6)
    x = torch.tanh(torch.randn(m, len(BSR_WIDTHS), h, generator=g))
    ws = [torch.randn(2 * d, h, generator=g) / h**0.5 for d in BSR_WIDTHS]
    bias = 0.1 * torch.randn(2 * sum(BSR_WIDTHS), generator=g)
    wall = torch.cat([w.reshape(-1) for w in ws]).cuda()
    _, pre = hip_ext.mask_estimator_final_forward_packed(x.cuda(), wall, bias.cuda(), BSR_WIDTHS)
    at = 0
    for b, d in enumerate(BSR_WIDTHS):
        if b in (0, 44, 61):
            cols = slice(2 * at, 2 * (at + d))
            assert torch.equal(pre[:, cols].cpu(), _chain(x[:, b], ws[b]) + bias[cols])
        at += d


@pytest.mark.parametrize("m,groups,i,o", [
    (99, 62, 192, 256),   # just above: the forward and dW split, dx (186 blocks of 128 rows) not
    (130, 62, 192, 256),  # all three
    (300, 62, 100, 260),  # columns, outputs and rows that end inside a tile, a partial K chunk each way
    (700, 62, 101, 140),  # widths no vector load fits: the forward alone
])
def test_large_products_keep_the_error_of_fp32_sums(hip_ext, m, groups, i, o):
    x, w, dy = (t.cuda() for t in _layer(m, groups, i, o, 7))
    _check_against_64_bits(hip_ext, x, w, dy)


def _check_against_64_bits(hip_ext, x, w, dy):
    (m, _, i), o = x.shape, w.shape[1]
    out = hip_ext.grouped_linear_forward(x, w)
    dx, dw, db = hip_ext.grouped_linear_backward(dy, x, w, True)
    xd, wd, dyd = x.double().transpose(0, 1).contiguous(), w.double(), dy.double().transpose(0, 1).contiguous()
    wt, dyt = wd.transpose(1, 2).contiguous(), dyd.transpose(1, 2).contiguous()
    exact = (torch.matmul(xd, wt).transpose(0, 1), torch.matmul(dyd, wd).transpose(0, 1), torch.matmul(dyt, xd))
    for got, want, k in zip((out, dx, dw), exact, (i, o, m)):
        rel = ((got.double() - want).norm() / want.norm()).item()
        assert rel <= 2.0**-23.5 * (1 + k**0.5 / 2), (rel, k)
    assert_parity(db, to_np(dyd.sum(1)), "f32", "db")


@pytest.mark.parametrize("exp", [-108, -112, -118, -124])
def test_numbers_too_small_for_bf16_parts(hip_ext, exp):
    """bf16 ends at 2^-133, so below 2^-110 three parts no longer hold 24 bits: 2^-118 lost 1e-5 of its
    value, also where a large weight makes the result an ordinary number."""
    x, w, dy = (t.cuda() for t in _layer(300, 62, 128, 260, 8))
    _check_against_64_bits(hip_ext, torch.ldexp(x, torch.tensor(exp)), torch.ldexp(w, torch.tensor(100)), dy)


def test_a_single_small_number(hip_ext):
    x, w, _ = (t.cuda() for t in _layer(300, 62, 128, 260, 8))
    clean = hip_ext.grouped_linear_forward(x, w)
    x[5, 3] = 0.0
    x[5, 3, 7] = 1.2345678 * 2.0**-121
    w2 = w.clone()
    w2[3, :, 7] *= 2.0**100
    out = hip_ext.grouped_linear_forward(x, w2)
    assert torch.equal(out[5, 3], x[5, 3, 7] * w2[3, :, 7])
    others = torch.arange(62) != 3
    assert torch.equal(out[:, others], clean[:, others])


@pytest.mark.parametrize("m,o", [(372, 192), (382, 192), (500, 260)])  # 0.293 G, 0.301 G, 0.53 G
def test_band_split_across_the_rule(hip_ext, m, o):
    _check_ragged(hip_ext, BSR_WIDTHS, m, o, torch.float32, 9)


@pytest.mark.parametrize("m", [142, 144, 200])  # 62 bands, hidden 256: 0.298 G, 0.302 G, 0.42 G
def test_mask_final_across_the_rule(hip_ext, m):
    h, dims = 256, BSR_WIDTHS
    g = torch.Generator().manual_seed(10)
    x = torch.tanh(torch.randn(m, len(dims), h, generator=g)).cuda()
    ws = [torch.randn(2 * d, h, generator=g) / h**0.5 for d in dims]
    wall = torch.cat([w.reshape(-1) for w in ws]).cuda()
    bias = (0.1 * torch.randn(2 * sum(dims), generator=g)).cuda()
    gout = torch.randn(m, sum(dims), generator=g).cuda()
    out, pre = hip_ext.mask_estimator_final_forward_packed(x, wall, bias, dims)
    npw = [to_np(w) for w in ws]
    r_out, r_pre = oracle.mask_estimator_final_forward(to_np(x), npw, to_np(bias), dims, "f32")[:2]
    assert_parity(out, r_out, "f32", "out")
    assert_parity(pre, r_pre, "f32", "pre")
    dz, db, dw = hip_ext.mask_estimator_final_backward_packed(gout, x, pre, wall, dims, input_activation="tanh")
    r_dz, r_db, r_dw = oracle.mask_estimator_final_backward(to_np(gout), to_np(x), to_np(pre), npw, dims, "f32",
                                                            input_act="tanh", grad_pre_dt="f32")
    assert_parity(dz, r_dz, "f32", "dz", by_index(1))
    assert_parity(db, r_db, "f32", "dbias", by_band(0, [2 * d for d in dims]))
    assert_parity(dw, np.concatenate([w.reshape(-1) for w in r_dw]), "f32", "dW")


@pytest.mark.parametrize("i,o", [(192, 192), (192, 256), (192, 128), (768, 320)])  # 12, 16, 8 and 16 tiles a wave
def test_forward_errors_have_no_sign(hip_ext, i, o):
    """The matrix cores cut off towards minus infinity.  The mean error of a result stays under 2^-28 of its
    RMS, a sixteenth of half a place (six products in one accumulator left 2^-26.5 at K = 192)."""
    x, w, _ = (t.cuda() for t in _layer(400, 62, i, o, 11))
    err = hip_ext.grouped_linear_forward(x, w).double().transpose(0, 1)
    want = torch.matmul(x.double().transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous())
    err = err - want
    assert abs(err.mean().item()) <= 2.0**-28 * want.pow(2).mean().sqrt().item()
    assert (err.norm() / want.norm()).item() <= 2.0**-23.5 * (1 + i**0.5 / 2)


def test_the_final_layers_errors_have_no_sign(hip_ext):
    m, h, dims = 400, 256, BSR_WIDTHS
    g = torch.Generator().manual_seed(12)
    x = torch.tanh(torch.randn(m, len(dims), h, generator=g)).cuda()
    ws = [(torch.randn(2 * d, h, generator=g) / h**0.5).cuda() for d in dims]
    bias = torch.zeros(2 * sum(dims), device="cuda")
    _, pre = hip_ext.mask_estimator_final_forward_packed(x, torch.cat([w.reshape(-1) for w in ws]), bias, dims)
    want = torch.cat([x[:, b].double() @ w.double().t().contiguous() for b, w in enumerate(ws)], 1)
    assert abs((pre.double() - want).mean().item()) <= 2.0**-28 * want.pow(2).mean().sqrt().item()


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_values_no_bf16_part_can_hold(hip_ext, bad):
    """3.4e38 rounds to infinity in bf16.  Row 5 of group 3 holds the value alone: the results are those of an
    fp32 product, other groups' are untouched, and the block that sums again counts every row of db once."""
    x, w, dy = (t.cuda() for t in _layer(300, 62, 128, 260, 13))
    clean = hip_ext.grouped_linear_forward(x, w)
    dx, dw, db = hip_ext.grouped_linear_backward(dy, x, w, True)
    x2 = x.clone()
    x2[5, 3] = 0.0
    x2[5, 3, 7] = bad
    out = hip_ext.grouped_linear_forward(x2, w)
    want = bad * w[3, :, 7]
    assert torch.equal(torch.isnan(out[5, 3]), torch.isnan(want))
    assert torch.equal(out[5, 3][~torch.isnan(want)], want[~torch.isnan(want)])
    others = torch.arange(62) != 3
    assert torch.equal(out[:, others], clean[:, others])
    rows = torch.arange(300) != 5
    assert torch.allclose(out[rows][:, 3], clean[rows][:, 3], rtol=1e-5, atol=1e-5)
    dy2 = dy.clone()
    dy2[5, 3, 11] = bad
    dx2, dw2, db2 = hip_ext.grouped_linear_backward(dy2, x, w, True)
    cols = torch.arange(260) != 11
    assert torch.equal(dx2[:, others], dx[:, others]) and torch.equal(dw2[others], dw[others])
    assert torch.equal(db2[3][cols], db[3][cols]) and torch.equal(db2[others], db[others])
    assert torch.allclose(dw2[3][cols], dw[3][cols], rtol=1e-4, atol=1e-4)
    assert bad == 3.4e38 or not torch.isfinite(db2[3, 11])


@pytest.mark.parametrize("bad", [float("inf"), 2.0**-125])
def test_row_norms_of_a_block_that_sums_again(hip_ext, bad):
    """The band split's forward gathers the rows' squares in its K loop: a weight that sends the block
    through it twice leaves inv_norm as it was."""
    m, o, dims = 400, 192, BSR_WIDTHS
    g = torch.Generator().manual_seed(14)
    x = torch.randn(m, sum(dims), generator=g).cuda()
    gamma = (1 + 0.1 * torch.randn(sum(dims), generator=g)).cuda()
    w = torch.cat([(torch.randn(o, d, generator=g) / d**0.5).reshape(-1) for d in dims]).cuda()
    b = torch.zeros(len(dims) * o, device="cuda")
    out, _, inv = hip_ext.band_split_ragged_forward_packed(x, gamma, w, b, dims, write_normed=False)
    w2 = w.clone()
    w2[o * sum(dims[:61]) + 3 * dims[61] + 100] = bad  # band 61, output 3
    out2, _, inv2 = hip_ext.band_split_ragged_forward_packed(x, gamma, w2, b, dims, write_normed=False)
    assert torch.equal(inv, inv2)
    assert torch.equal(out[:, :61], out2[:, :61])
    cols = torch.arange(o) != 3
    assert torch.allclose(out[:, 61][:, cols], out2[:, 61][:, cols], rtol=1e-4, atol=1e-5)
    assert bad < 1 or not torch.isfinite(out2[:, 61, 3]).any()
