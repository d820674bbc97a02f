"""The work this package is measured on: its fused layers at the sizes its users train with.

A case is one pass, forward and backward, through one layer of a band-split or mel-band RoFormer
(``kind``), called as the patched training step calls it, plus one whole training step of the tiny
model.  Sizes are those of the training configurations in ``pymsst_amd.workloads`` (and, for
``draw``, what lies between and around them):

* rows ``m`` = batch x frames: 130 (tiny), 1032 (BS-RoFormer), 1896 (dim 512), 2760 (mel);
* ``dim`` / ``hidden``: 64 / 256, 192 / 768, 512 / 2048, and other multiples of 32;
* bands: the 62 BS-RoFormer bands (4100 stereo features), the 60 overlapping mel bands (7916), mono
  halves of both, and a short list of odd widths;
* fp32 without autocast, bf16 or fp16 with it.

Every tensor a backward needs is kept from the forward, and each pass returns the layer's output and
all of its gradients.
"""

from __future__ import annotations

import os

import torch

from pymsst_amd import fused_roformer as fr
from pymsst_amd.core.bs_roformer import DEFAULT_FREQS_PER_BANDS
from pymsst_amd.core.mel_band_roformer import mel_band_bins
from pymsst_amd.core.transformer import RotaryEmbedding
from pymsst_amd.fused_extension import load_fused_band_split_extension
from pymsst_amd.workloads import WORKLOADS, workload_batch

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_ODD = (3, 5, 2, 7, 33, 9, 65, 130)  # real + imaginary parts of no whole bin: widths no vector load fits


def listed():
    return [
        # the first layer of the tiny fp32 model: a call whose launches are most of its time
        dict(name="band_split_tiny_fp32", kind="band_split", bands="bsr", channels=2, m=130, dim=64, dtype="fp32"),
        # the first layer of BS-RoFormer training: fp32 spectrum in, bf16 projection out
        dict(name="band_split_bsr_bf16", kind="band_split", bands="bsr", channels=2, m=1032, dim=192, dtype="bf16"),
        # the same of the Mel-band model: its bands overlap and its clips are longer
        dict(name="band_split_mel_bf16", kind="band_split", bands="mel", channels=2, m=2760, dim=192, dtype="bf16"),
        # the mask estimator of the tiny fp32 model
        dict(name="mask_mlp_tiny_fp32", kind="mask_mlp", bands="bsr", channels=2, m=130, dim=64, hidden=256,
             dtype="fp32"),
        # the mask estimator of BS-RoFormer training without autocast
        dict(name="mask_mlp_bsr_fp32", kind="mask_mlp", bands="bsr", channels=2, m=1032, dim=192, hidden=768,
             dtype="fp32"),
        # the mask estimators of BS-RoFormer training with their mask product: four stems of a batch of 4
        dict(name="mask_core_bsr_bf16", kind="mask_core", bands="bsr", channels=2, batch=4, frames=258, stems=4,
             dim=192, hidden=768, dtype="bf16"),
        # the mask estimator of the Mel-band model, in fp16 (training with a loss scaler)
        dict(name="mask_mlp_mel_fp16", kind="mask_mlp", bands="mel", channels=2, m=2760, dim=192, hidden=768,
             dtype="fp16"),
        # the mask estimator of the dim-512 model: the largest layer
        dict(name="mask_mlp_dim512_bf16", kind="mask_mlp", bands="bsr", channels=2, m=1896, dim=512, hidden=2048,
             dtype="bf16"),
        # the norm in front of every attention and feed-forward of BS-RoFormer training
        dict(name="rms_norm_bsr_bf16", kind="rms_norm", rows=63984, dim=192, dtype="bf16"),
        # q/k norm and rotary over the time axis of BS-RoFormer training
        dict(name="qk_norm_rotary_bsr_bf16", kind="qk_norm_rotary", batch=248, n=258, heads=8, head_dim=64,
             dtype="bf16"),
        # what surrounds attention in the dim-512 model: qkv split + rotary, output gate
        dict(name="attention_io_dim512_bf16", kind="attention_io", batch=124, n=948, heads=8, head_dim=64, dim=512,
             dtype="bf16"),
        # a whole training step (loss, gradients) of the tiny model: many small calls, the host in between
        dict(name="train_step_tiny_fp32", kind="train_step", dtype="fp32"),
    ]


def draw(rng):
    kind = rng.choice(["band_split", "band_split", "mask_mlp", "mask_mlp", "mask_mlp", "mask_core", "rms_norm",
                       "qk_norm_rotary", "attention_io"])
    dtype = rng.choice(["fp32", "bf16", "bf16", "fp16"])

    def logint(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    bands = rng.choice(["bsr", "bsr", "mel", "mel", "odd"])
    channels = rng.choice([1, 2, 2])
    if kind == "band_split":
        return dict(kind=kind, bands=bands, channels=channels, m=logint(31, 3000),
                    dim=rng.choice([64, 96, 128, 192, 256, 384, 512]), dtype=dtype)
    if kind in ("mask_mlp", "mask_core"):
        if dtype != "fp32":  # 16-bit estimators are trained on stereo models: widths in whole fours
            bands, channels = "bsr" if bands == "odd" else bands, 2
        dim = rng.choice([64, 96, 128, 192, 192, 256, 384, 512])
        hidden = dim * rng.choice([2, 4, 4])
        # no dearer than the largest listed case (fp32 and 60 wide mel bands cost more a row)
        most = min(3000, 1896 * 512 * 2048 // (dim * hidden) // (4 if dtype == "fp32" else 2 if bands == "mel" else 1))
        if kind == "mask_mlp":
            return dict(kind=kind, bands=bands, channels=channels, m=logint(31, max(most, 64)), dim=dim, hidden=hidden,
                        dtype=dtype)
        stems, batch = rng.choice([1, 2, 4]), rng.choice([1, 2, 3, 4])
        dtype, channels = "bf16" if dtype == "fp32" else dtype, 2  # the mask product is fused in 16 bits
        most = 1896 * 512 * 2048 // (dim * hidden) // 2
        return dict(kind=kind, bands="bsr", channels=channels, batch=batch,
                    frames=logint(17, max(min(1200, most // stems) // batch, 32)), stems=stems, dim=dim, hidden=hidden,
                    dtype=dtype)
    if kind == "rms_norm":
        dim = rng.choice([64, 96, 128, 192, 256, 384, 512])
        return dict(kind=kind, rows=logint(1000, 120000 * 192 // dim), dim=dim, dtype=dtype)
    n, heads, head_dim = logint(31, 1000), rng.choice([4, 8]), rng.choice([32, 64])
    batch = max(1, logint(4, 124 * 948) // n)
    if kind == "qk_norm_rotary":
        return dict(kind=kind, batch=batch, n=n, heads=heads, head_dim=head_dim, dtype=dtype)
    return dict(kind=kind, batch=batch, n=n, heads=heads, head_dim=head_dim,
                dim=rng.choice([64, 128, 192, 256, 384, 512]), dtype=dtype)


# ---------------------------------------------------------------------- inputs


def _widths(case):
    if case["bands"] == "odd":
        return _ODD * 4
    bins = DEFAULT_FREQS_PER_BANDS if case["bands"] == "bsr" else [len(b) for b in mel_band_bins(44100, 2048, 60)]
    return tuple(2 * case["channels"] * int(b) for b in bins)


class _Inputs:
    """Seeded normal tensors on the GPU, rounded to the dtype the layer gets them in."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def __call__(self, *shape, scale=1.0, shift=0.0, dtype=None):
        t = torch.randn(*shape, generator=self.gen, device="cuda")
        return t.mul_(scale).add_(shift).to(dtype or self.dtype)


def _packed_weights(rand, rows_of, cols_of, widths):
    """One ``[rows, cols]`` matrix per band, uniform variance 1 / cols, back to back."""
    return torch.cat([rand(rows_of(w), cols_of(w), scale=cols_of(w) ** -0.5).reshape(-1) for w in widths])


def _inputs(case, seed):
    """The tensors of a case, by name (the same for ``run`` and for ``exact``)."""
    kind, dt = case["kind"], _DTYPES[case["dtype"]]
    rand = _Inputs(seed, dt)
    t = {}
    if kind == "band_split":
        w = _widths(case)
        m, total, nb, dim = case["m"], sum(w), len(w), case["dim"]
        # a spectrum: fp32 whatever the projection's type, each bin of its own size
        t["x"] = rand(m, total, dtype=torch.float32) * torch.exp(rand(1, total, dtype=torch.float32))
        t["gamma"] = rand(total, scale=0.1, shift=1.0, dtype=torch.float32)
        t["weight"] = _packed_weights(rand, lambda i: dim, lambda i: i, w)
        t["bias"] = rand(nb * dim, scale=0.1)
        t["grad_out"] = rand(m, nb, dim)
    elif kind in ("mask_mlp", "mask_core"):
        w = _widths(case)
        total, nb, dim, hidden = sum(w), len(w), case["dim"], case["hidden"]
        m = case["m"] if kind == "mask_mlp" else case["batch"] * case["frames"]
        t["x"] = rand(m, nb, dim)  # behind the final norm
        for s in range(1 if kind == "mask_mlp" else case["stems"]):
            t["w1_%d" % s] = rand(nb, hidden, dim, scale=dim ** -0.5)
            t["b1_%d" % s] = rand(nb, hidden, scale=0.1)
            t["w2_%d" % s] = _packed_weights(rand, lambda i: 2 * i, lambda i: hidden, w)
            t["b2_%d" % s] = rand(2 * total, scale=0.1)
        if kind == "mask_mlp":
            t["grad_out"] = rand(m, total)
        else:
            b, n, s, c = case["batch"], case["frames"], case["stems"], case["channels"]
            t["spec"] = torch.view_as_complex(rand(b, total // 2, n, 2, dtype=torch.float32))
            t["grad_est"] = torch.view_as_complex(rand(b * s * c, total // 2 // c, n, 2, dtype=torch.float32))
    elif kind == "rms_norm":
        t["x"] = rand(case["rows"], case["dim"], scale=2.0)
        t["gamma"] = rand(case["dim"], scale=0.1, shift=1.0, dtype=torch.float32)
        t["grad_out"] = rand(case["rows"], case["dim"])
    elif kind in ("qk_norm_rotary", "attention_io"):
        b, n, h, d = case["batch"], case["n"], case["heads"], case["head_dim"]
        cos, sin = RotaryEmbedding(d, 10000.0).tables(n, torch.device("cuda"), dt)
        t["cos"], t["sin"] = cos[..., ::2], sin[..., ::2]
        if kind == "qk_norm_rotary":
            for name in ("q", "k", "grad_q", "grad_k"):
                t[name] = rand(b, n, h, d)
            t["gamma_q"] = rand(d, scale=0.1, shift=1.0, dtype=torch.float32)
            t["gamma_k"] = rand(d, scale=0.1, shift=1.0, dtype=torch.float32)
        else:
            t["qkv"] = rand(b, n, 3 * h * d)
            # as attention gives them: dense [b, n, h, d] in 16 bits, a transpose of [b, h, n, d] in fp32
            for name in ("grad_q", "grad_k", "grad_v", "attn"):
                t[name] = rand(b, h, n, d).transpose(1, 2) if dt == torch.float32 else rand(b, n, h, d)
            t["x"] = rand(b * n, case["dim"])
            t["weight"] = rand(h, case["dim"], scale=case["dim"] ** -0.5)
            t["bias"] = rand(h, scale=0.1)
            t["grad_out"] = rand(b * n, h * d)
    return t


def prepare(case, seed):
    if case["kind"] == "train_step":
        return _prepare_train_step(case, seed)
    state = dict(case, ext=load_fused_band_split_extension(), **_inputs(case, seed))
    if "bands" in case:
        state["widths"] = _widths(case)
    return state


def _prepare_train_step(case, seed):
    os.environ.update(fr.RUNTIME_PRESETS["hip_full"])
    workload = WORKLOADS["bsr_tiny"]
    model = workload.build_model(torch.device("cuda"), seed=seed)
    model.train()
    fr.apply_roformer_fused_training_backend(model, "hip", rms_norm_mode="fast")
    target, mixture = workload_batch(workload, seed=seed, device=torch.device("cuda"))
    return dict(kind="train_step", model=model, target=target, mixture=mixture)


# ---------------------------------------------------------------------- one pass


def run(state):
    return _RUN[state["kind"]](state)


def _run_band_split(s):
    ext, w = s["ext"], s["widths"]
    if s["dtype"] == "fp32":
        out, _, inv = ext.band_split_ragged_forward_packed(s["x"], s["gamma"], s["weight"], s["bias"], w,
                                                           write_normed=False)
        grads = ext.band_split_ragged_backward_packed(s["grad_out"], s["x"], True, inv, s["gamma"], s["weight"], w)
    else:
        out, feats, inv = ext.band_split_mixed_forward(s["x"], s["gamma"], s["weight"], s["bias"], w,
                                                       s["weight"].dtype)
        grads = ext.band_split_mixed_backward(s["grad_out"], s["x"], feats, inv, s["gamma"], s["weight"], w)
    return [out, *grads]


def _run_mask_mlp(s):
    ext, w = s["ext"], s["widths"]
    x, w1, b1, w2, b2 = s["x"], s["w1_0"], s["b1_0"], s["w2_0"], s["b2_0"]
    if ext.mask_mlp_supported(x.shape[-1], w1.shape[1], w, x.dtype):
        out, pre, hidden = ext.mask_mlp_forward(x, w1, b1, w2, b2, w, save_hidden=True)
    else:
        hidden = ext.grouped_linear_forward_act(x, w1, b1, activation="tanh")
        out, pre = ext.mask_estimator_final_forward_packed(hidden, w2, b2, w)
    dz, db2, dw2 = ext.mask_estimator_final_backward_packed(s["grad_out"], hidden, pre, w2, w, input_activation="tanh")
    dx, dw1, db1 = ext.grouped_linear_backward(dz, x, w1)
    return [out, dx, dw1, db1, dw2, db2]


def _run_mask_core(s):
    ext, w, stems, channels = s["ext"], s["widths"], s["stems"], s["channels"]
    x, spec = s["x"], s["spec"]
    fused = ext.mask_mlp_supported(x.shape[-1], s["hidden"], w, x.dtype)
    b, fc, t = spec.shape
    saved, masks = [], []
    if fused:
        est = torch.empty((b * stems * channels, fc // channels, t), dtype=torch.complex64, device=x.device)
    for i in range(stems):
        w1, b1, w2, b2 = (s["%s_%d" % (n, i)] for n in ("w1", "b1", "w2", "b2"))
        if fused:
            pre, hidden = ext.mask_mlp_forward_apply(x, w1, b1, w2, b2, w, spec, est, i, channels, save_hidden=True)
        else:
            hidden = ext.grouped_linear_forward_act(x, w1, b1, activation="tanh")
            mask, pre = ext.mask_estimator_final_forward_packed(hidden, w2, b2, w)
            masks.append(mask.view(b, t, 2 * fc))
        saved.append((w1, hidden, pre, w2))
    if not fused:
        est = ext.mask_apply_forward(spec, torch.stack(masks, dim=1), channels)
    grad_mask = ext.mask_apply_grad_mask(s["grad_est"], spec, stems, channels, x.dtype)
    dx, grads = None, []
    for i, (w1, hidden, pre, w2) in enumerate(saved):
        g = grad_mask[:, i].reshape(x.shape[0], -1)
        dz, db2, dw2 = ext.mask_estimator_final_backward_packed(g, hidden, pre, w2, w, input_activation="tanh")
        dxi, dw1, db1 = ext.grouped_linear_backward(dz, x, w1)
        dx = dxi if dx is None else dx + dxi
        grads += [dw1, db1, dw2, db2]
    return [est, dx, *grads]


def _run_rms_norm(s):
    out, inv = s["ext"].rms_norm_forward_lean(s["x"], s["gamma"])
    return [out, *s["ext"].rms_norm_backward_from_input(s["grad_out"], s["x"], inv, s["gamma"])]


def _run_qk_norm_rotary(s):
    qo, ko, inv_q, inv_k = s["ext"].rms_norm_rotary_pair_forward(s["q"], s["k"], s["gamma_q"], s["gamma_k"], s["cos"],
                                                                 s["sin"])
    return [qo, ko, *s["ext"].rms_norm_rotary_pair_backward(s["grad_q"], s["grad_k"], s["q"], s["k"], inv_q, inv_k,
                                                            s["gamma_q"], s["gamma_k"], s["cos"], s["sin"])]


def _run_attention_io(s):
    ext = s["ext"]
    layout = "bhnd" if s["dtype"] == "fp32" else "bnhd"  # what attention reads in each type
    q, k, v = ext.rotary_qkv_forward(s["qkv"], s["heads"], s["cos"], s["sin"], out_layout=layout)
    out, gate, attn, x = ext.attention_gate_forward_bnhd(s["attn"], s["x"], s["weight"], s["bias"])
    grads = ext.attention_gate_backward_bnhd(s["grad_out"], attn, x, s["weight"], gate, out_layout=layout)
    dqkv = ext.rotary_qkv_backward(s["grad_q"], s["grad_k"], s["grad_v"], s["cos"], s["sin"])
    return [q, k, v, out, *grads, dqkv]


def _run_train_step(s):
    model = s["model"]
    loss = model(s["mixture"], s["target"])
    loss.backward()
    grads = torch.cat([p.grad.reshape(-1) for p in model.parameters()])
    model.zero_grad(set_to_none=True)
    return [loss.detach(), grads]


_RUN = {"band_split": _run_band_split, "mask_mlp": _run_mask_mlp, "mask_core": _run_mask_core,
        "rms_norm": _run_rms_norm, "qk_norm_rotary": _run_qk_norm_rotary, "attention_io": _run_attention_io,
        "train_step": _run_train_step}


# ---------------------------------------------------------------------- what a pass cannot do without


def work(case):
    """Bytes: the layer's inputs (activations, parameters, incoming gradient) read once and its outputs
    and gradients written once.  Flops: its matrix products, forward and backward."""
    kind = case["kind"]
    s = 4 if case["dtype"] == "fp32" else 2
    if kind == "band_split":
        w = _widths(case)
        m, total, nb, dim = case["m"], sum(w), len(w), case["dim"]
        params = total * dim + nb * dim
        return {"bytes": 2 * m * total * 4 + 2 * total * 4 + 2 * params * s + 2 * m * nb * dim * s,
                "flops": 6 * m * total * dim}
    if kind in ("mask_mlp", "mask_core"):
        w = _widths(case)
        total, nb, dim, hidden = sum(w), len(w), case["dim"], case["hidden"]
        stems = case.get("stems", 1)
        m = case["m"] if kind == "mask_mlp" else case["batch"] * case["frames"]
        params = stems * (nb * hidden * (dim + 1) + 2 * total * (hidden + 1))
        acts = 2 * m * nb * dim * s + (2 * m * total * s if kind == "mask_mlp" else (1 + 2 * stems) * m * total * 4)
        return {"bytes": acts + 2 * params * s, "flops": 6 * stems * m * (nb * dim * hidden + 2 * total * hidden)}
    if kind == "rms_norm":
        return {"bytes": 4 * case["rows"] * case["dim"] * s + 8 * case["dim"], "flops": 0}
    if kind in ("qk_norm_rotary", "attention_io"):
        rows, hd = case["batch"] * case["n"], case["heads"] * case["head_dim"]
        if kind == "qk_norm_rotary":
            return {"bytes": 8 * rows * hd * s, "flops": 0}
        gate = rows * (4 * hd + 2 * case["dim"]) * s
        return {"bytes": 12 * rows * hd * s + gate, "flops": 6 * rows * case["heads"] * case["dim"]}
    workload = WORKLOADS["bsr_tiny"]
    w, dim = [4 * f for f in DEFAULT_FREQS_PER_BANDS], workload.model["dim"]
    m, total, nb, inner = 130, sum(w), len(w), workload.model["heads"] * workload.model["dim_head"]
    mlp = nb * dim * 4 * dim + 2 * total * 4 * dim
    block = 4 * dim * inner + 8 * dim * dim
    params = total * dim + mlp + 2 * block
    return {"bytes": 8 * params + 4 * 2 * 2 * 2 * 32768, "flops": 6 * m * (total * dim + mlp + 2 * nb * block)}


def tolerance(case):
    """About four times what the layers are off their 64-bit results, over the listed cases and two dozen
    drawn ones: fp32 up to 8e-7 (largest element 1.1e-5), bf16 5.2e-3 (0.06), fp16 6.5e-4 (7e-3).  The
    training step chains two dozen layers."""
    if case["kind"] == "train_step":
        return {"rel": 2e-5, "max": 1e-3}
    return {"fp32": {"rel": 4e-6, "max": 5e-5}, "bf16": {"rel": 2e-2, "max": 0.25},
            "fp16": {"rel": 2.6e-3, "max": 0.03}}[case["dtype"]]


# ---------------------------------------------------------------------- the same in 64 bits


def exact(case, seed):
    if case["kind"] == "train_step":
        return None
    t = {k: (v.to(torch.complex128) if v.is_complex() else v.double()) for k, v in _inputs(case, seed).items()}
    return _EXACT[case["kind"]](case, t)


def _norm_backward(dy, x, inv, gamma):
    """Gradients of ``x * inv * sqrt(D) * gamma``."""
    root = x.shape[-1] ** 0.5
    n = x * inv * root
    t = dy * gamma
    dx = inv * (t * root - n * (t * n).sum(-1, keepdim=True) / root)
    return dx, (dy * n).sum(0)


def _exact_band_split(case, t):
    widths, dim = _widths(case), case["dim"]
    outs, dxs, dgs, dws, dbs = [], [], [], [], []
    at = 0
    for b, i in enumerate(widths):
        x, gamma = t["x"][:, at:at + i], t["gamma"][at:at + i]
        weight = t["weight"][dim * at:dim * (at + i)].view(dim, i)
        inv = 1.0 / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        f = x * inv * i ** 0.5 * gamma
        dy = t["grad_out"][:, b].contiguous()
        outs.append(f @ weight.t().contiguous() + t["bias"][b * dim:(b + 1) * dim])
        dx, dg = _norm_backward(dy @ weight, x, inv, gamma)
        dxs.append(dx)
        dgs.append(dg)
        dws.append((dy.t().contiguous() @ f).reshape(-1))
        dbs.append(dy.sum(0))
        at += i
    return [torch.stack(outs, 1), torch.cat(dxs, 1), torch.cat(dgs), torch.cat(dws), torch.cat(dbs)]


def _exact_mlp(case, t, stem, grad_out):
    """``(mask, dx, dw1, db1, dw2, db2)`` of one estimator; ``grad_out`` is the mask's gradient."""
    widths, hidden = _widths(case), case["hidden"]
    x, w1, b1, w2, b2 = t["x"], *(t["%s_%d" % (n, stem)] for n in ("w1", "b1", "w2", "b2"))
    dx, dw1, db1 = torch.empty_like(x), torch.empty_like(w1), torch.empty_like(b1)
    outs, dw2s, db2s = [], [], []
    at = 0
    for b, i in enumerate(widths):
        xb, w2b = x[:, b].contiguous(), w2[2 * at * hidden:2 * (at + i) * hidden].view(2 * i, hidden)
        h = torch.tanh(xb @ w1[b].t().contiguous() + b1[b])
        pre = h @ w2b.t().contiguous() + b2[2 * at:2 * (at + i)]
        left, gate = pre[:, :i], torch.sigmoid(pre[:, i:])
        outs.append(left * gate)
        g = grad_out[:, at:at + i]
        dpre = torch.cat([g * gate, g * left * gate * (1 - gate)], 1)
        dw2s.append((dpre.t().contiguous() @ h).reshape(-1))
        db2s.append(dpre.sum(0))
        dz = (dpre @ w2b) * (1 - h * h)
        dx[:, b] = dz @ w1[b]
        dw1[b] = dz.t().contiguous() @ xb
        db1[b] = dz.sum(0)
        at += i
    return torch.cat(outs, 1), dx, dw1, db1, torch.cat(dw2s), torch.cat(db2s)


def _exact_mask_mlp(case, t):
    return list(_exact_mlp(case, t, 0, t["grad_out"]))


def _exact_mask_core(case, t):
    b, n, stems, c = case["batch"], case["frames"], case["stems"], case["channels"]
    spec = t["spec"]
    fc = spec.shape[1]
    grad = t["grad_est"].view(b, stems, c, fc // c, n).transpose(2, 3).reshape(b, stems, fc, n)
    est, dx, grads = [], 0, []
    for s in range(stems):
        g = torch.view_as_real((grad[:, s] * spec.conj()).resolve_conj().transpose(1, 2).contiguous())
        mask, dxs, dw1, db1, dw2, db2 = _exact_mlp(case, t, s, g.reshape(b * n, 2 * fc))
        dx = dx + dxs
        grads += [dw1, db1, dw2, db2]
        est.append(spec * torch.view_as_complex(mask.view(b, n, fc, 2)).transpose(1, 2))
    est = torch.stack(est, 1).view(b, stems, fc // c, c, n).transpose(2, 3).reshape(b * stems * c, fc // c, n)
    return [est.contiguous(), dx, *grads]


def _exact_rms_norm(case, t):
    inv = 1.0 / t["x"].norm(dim=-1, keepdim=True).clamp_min(1e-12)
    return [t["x"] * inv * case["dim"] ** 0.5 * t["gamma"], *_norm_backward(t["grad_out"], t["x"], inv, t["gamma"])]


def _rotate(x, cos, sin):
    """Pairs (2p, 2p + 1) of the last axis turned by the angle of their position and pair."""
    a, b = x[..., ::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)


def _exact_qk_norm_rotary(case, t):
    outs, grads, gammas = [], [], []
    for n in ("q", "k"):
        x, gamma = t[n], t["gamma_" + n]
        inv = 1.0 / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        outs.append(_rotate(x * inv * x.shape[-1] ** 0.5 * gamma, t["cos"], t["sin"]))
        dx, dg = _norm_backward(_rotate(t["grad_" + n], t["cos"], -t["sin"]), x, inv, gamma)
        grads.append(dx)
        gammas.append(dg.sum((0, 1)))
    return [*outs, *grads, *gammas]


def _exact_attention_io(case, t):
    b, n, h, d = case["batch"], case["n"], case["heads"], case["head_dim"]
    q, k, v = t["qkv"].view(b, n, 3, h, d).unbind(2)
    cos, sin = t["cos"], t["sin"]
    gate = torch.sigmoid(t["x"] @ t["weight"].t().contiguous() + t["bias"])
    attn, grad = t["attn"].reshape(-1, h, d), t["grad_out"].view(-1, h, d)
    gpre = (attn * grad).sum(-1) * gate * (1 - gate)
    dqkv = torch.stack([_rotate(t["grad_q"], cos, -sin), _rotate(t["grad_k"], cos, -sin), t["grad_v"]], 2)
    return [_rotate(q, cos, sin), _rotate(k, cos, sin), v, (attn * gate[..., None]).reshape(b * n, h * d),
            (grad * gate[..., None]).reshape(b, n, h, d), gpre @ t["weight"], gpre.t().contiguous() @ t["x"], gpre.sum(0),
            dqkv.view(b, n, 3 * h * d)]


_EXACT = {"band_split": _exact_band_split, "mask_mlp": _exact_mask_mlp, "mask_core": _exact_mask_core,
          "rms_norm": _exact_rms_norm, "qk_norm_rotary": _exact_qk_norm_rotary, "attention_io": _exact_attention_io}
