"""The work that a program built on ``hstu_amd`` has it do, as cases to time.

A case is one pass through the package's public entry points: jagged attention
(scoring, and training with its backward), the projection GEMMs, the output
block's LayerNorm, the targets-only last layer and the whole HSTU layer, in
bf16 and in e4m3, from a handful of short sequences to the full training
batch.  ``listed`` holds the fixed ones, ``draw`` gives more of the same
ranges; ``prepare`` / ``run`` are the program's set-up and one pass, ``exact``
the same results in 64 bits from plain torch.
"""

import math
import os
import sys

# The training job's environment: the FP8 P.V forward, the full-FP8 attention
# backward with its dS pre-scale, and the 16-bit dropout masks.
os.environ["DLRM_HSTU_FP8_FWD_PV"] = "1"
os.environ["DLRM_HSTU_FP8_BWD_FULL"] = "1"
os.environ["DLRM_HSTU_FP8_BWD_FULL_DSC_K"] = "-5"
os.environ["DLRM_HSTU_FP8_MASK16"] = "1"
sys.path.insert(1, os.path.join(os.getcwd(), "mlperf-training_amd"))

import numpy as np  # noqa: E402
import torch  # noqa: E402

import hstu_amd  # noqa: E402
from hstu_amd import bwd_fp8, fp8  # noqa: E402

E4M3 = torch.float8_e4m3fn
WIDTH = 512          # embedding width E = H * D of the layer
MAX_TOKENS = 162251  # tokens of the full training batch
MAX_PAIRS = 300720505  # its causal (query, key) pairs per head
DROPOUT, DROPOUT_SEED = 0.3, 11
EPS = 1e-6


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # scoring a few short histories: one forward call, where latency counts
        dict(name="attn_fwd_short", path="attention", dtype="bf16", train=False, heads=2, dim=64, mask="causal",
             lengths="uniform", batch=8, low=16, high=256, max_len=256, length_seed=0),
        # scoring candidates for one user with a long history: one sequence, its last rows are targets
        dict(name="attn_fwd_one_user", path="attention", dtype="bf16", train=False, heads=4, dim=128, mask="targets",
             lengths="uniform", batch=1, low=3001, high=3001, max_len=4096, length_seed=0),
        # the forward of a medium batch with a learned relative-position bias
        dict(name="attn_fwd_bias", path="attention", dtype="bf16", train=False, heads=4, dim=128, mask="bias",
             lengths="uniform", batch=64, low=128, high=1024, max_len=1024, length_seed=0),
        # training attention with ranking targets, a local window and a contextual prefix
        dict(name="attn_train_masks", path="attention", dtype="bf16", train=True, heads=4, dim=128, mask="all",
             lengths="uniform", batch=64, low=128, high=1024, max_len=1024, length_seed=0),
        # training attention of the full long-tailed batch in bf16
        dict(name="attn_train_bf16", path="attention", dtype="bf16", train=True, heads=4, dim=128, mask="bias",
             lengths="zipf", batch=128, low=32, high=4096, max_len=4096, length_seed=0),
        # the same batch in e4m3 with per-(token, head) scales
        dict(name="attn_train_fp8", path="attention", dtype="e4m3", train=True, heads=4, dim=128, mask="bias",
             lengths="zipf", batch=128, low=32, high=4096, max_len=4096, length_seed=0),
        # the last layer, where only one target row of each sequence attends, forward and backward
        dict(name="targets_only_train", path="delta", dtype="e4m3", heads=4, dim=128, rows=1,
             lengths="zipf", batch=128, low=32, high=4096, max_len=4096, length_seed=0),
        # the UVQK projection of a full batch, SiLU on its U columns
        dict(name="gemm_uvqk_fp8", path="gemm", m=262144, n=2048, k=512, silu=512, residual=False),
        # the output projection of a small scoring batch
        dict(name="gemm_out_small", path="gemm", m=1027, n=512, k=1536, silu=0, residual=True),
        # the output block's LayerNorm * U * dropout of a full batch, forward and backward
        dict(name="norm_mul_dropout", path="norm", tokens=MAX_TOKENS),
        # a training step of one layer in bf16 on a medium batch
        dict(name="layer_train_bf16", path="layer", dtype="bf16", lengths="uniform", batch=64, low=128, high=1024,
             max_len=1024, length_seed=0),
        # a training step of one layer in FP8 on the full batch
        dict(name="layer_train_fp8", path="layer", dtype="e4m3", lengths="zipf", batch=128, low=32, high=4096,
             max_len=4096, length_seed=0),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_lengths(rng, max_len_low, max_len_high):
    """Sequences within the full batch's tokens and pairs."""
    while True:
        max_len = _log_int(rng, max_len_low, max_len_high)
        c = dict(lengths=rng.choice(["uniform", "zipf"]), batch=_log_int(rng, 1, 128),
                 low=max(4, max_len // 32), high=max_len, max_len=max_len, length_seed=rng.randrange(1000))
        lens = _lengths(c)
        if lens.sum() <= MAX_TOKENS and _pairs(lens) <= MAX_PAIRS:
            return c


def draw(rng):
    path = rng.choice(["attention"] * 5 + ["delta", "gemm", "gemm", "norm", "layer", "layer"])
    if path == "attention":
        dtype = rng.choice(["bf16", "bf16", "e4m3"])
        dim = 128 if dtype == "e4m3" else rng.choice([64, 128])
        return dict(path=path, dtype=dtype, train=rng.random() < 0.6, heads=rng.choice([1, 2, 4]), dim=dim,
                    mask=rng.choice(["causal", "bias", "targets", "all"]), **_draw_lengths(rng, 64, 6000))
    if path == "delta":
        return dict(path=path, dtype=rng.choice(["bf16", "e4m3"]), heads=rng.choice([2, 4]), dim=128,
                    rows=rng.choice([1, 1, 2, 4]), **_draw_lengths(rng, 128, 6000))
    if path == "gemm":
        m = _log_int(rng, 33, 262144)
        if rng.random() < 0.5:
            n = rng.choice([512, 1536, 2048])
            return dict(path=path, m=m, n=n, k=512, silu=rng.choice([0, 512]), residual=False)
        return dict(path=path, m=m, n=512, k=1536, silu=0, residual=True)
    if path == "norm":
        return dict(path=path, tokens=_log_int(rng, 100, MAX_TOKENS))
    return dict(path=path, dtype=rng.choice(["bf16", "e4m3"]), **_draw_lengths(rng, 64, 4096))


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _lengths(c):
    rng = np.random.default_rng(c["length_seed"])
    if c["lengths"] == "zipf":
        return rng.zipf(1.2, c["batch"]).clip(c["low"], c["high"]).astype(np.int64)
    return rng.integers(c["low"], c["high"] + 1, c["batch"]).astype(np.int64)


def _pairs(lens):
    return int((lens * (lens + 1) // 2).sum())


def _mask_options(c, lens):
    """(num_targets [B] or None, window, contextual prefix) of a case's mask."""
    if c.get("mask") not in ("targets", "all"):
        return None, 0, 0
    rng = np.random.default_rng(c["length_seed"] + 1)
    high = max(1, min(64, int(lens.min()) // 4))
    nt = rng.integers(1, high + 1, len(lens)).astype(np.int32)
    return (nt, max(8, c["max_len"] // 4), 3) if c["mask"] == "all" else (nt, 0, 0)


def _bias_span(c):
    return min(c["max_len"], 1024)


def _valid(length, nt, window, prefix, device):
    """The mask of one sequence: causal on positions where the prefix and the
    targets each share one, a window, and prefix rows that see the history."""
    pos = torch.arange(length, device=device)
    last = length
    if prefix > 0:
        pos = (pos - prefix + 1).clamp_min(0)
        last = last - prefix + 1
    if nt is not None:
        last = last - nt
        pos = pos.clamp_max(last)
    dist = pos[:, None] - pos[None, :]
    valid = (dist > 0) | torch.eye(length, dtype=torch.bool, device=device)
    if window > 0:
        valid &= dist <= window
    if prefix > 0:
        valid |= (pos[:, None] == 0) & (pos[None, :] < last)
    return valid


def _valid_pairs(c, lens):
    nt, window, prefix = _mask_options(c, lens)
    if nt is None:
        return _pairs(lens)
    total = 0
    for b, length in enumerate(lens.tolist()):
        last = length - (prefix - 1 if prefix else 0) - int(nt[b])  # history positions
        p = np.minimum(np.arange(length) - (prefix - 1 if prefix else 0), last).clip(0)
        seen = p if window == 0 else np.minimum(p, window)
        if prefix:
            seen = np.where(p == 0, last + prefix - 2, seen + np.where(p <= window, prefix - 1, 0))
        total += int((seen + 1).sum())
    return total


def _attention_work(c, lens):
    T, H, D = int(lens.sum()), c["heads"], c["dim"]
    es = 1 if c["dtype"] == "e4m3" else 2
    pairs = _valid_pairs(c, lens)
    nbytes = T * H * D * (3 * es + 2) + (12 * T * H if es == 1 else 0)
    flops = 4 * D * H * pairs
    if c["train"]:
        nbytes += T * H * D * (2 + 6)
        flops += 10 * D * H * pairs
    return nbytes, flops


def work(c):
    if c["path"] == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": m * k + n * k + 2 * m * n * (2 if c["residual"] else 1) + 4 * m + 6 * n,
                "flops": 2 * m * n * k}
    if c["path"] == "norm":
        D = WIDTH
        fwd = 2 * D + 2 * D + 3 * D + D + 8          # x, u in; e4m3 y, mask, statistics out
        bwd = 6 * D + 4 * D + D + 8 + 4 * D + 6 * D  # dy, x, u, mask, statistics in; dx, du, y out
        return {"bytes": c["tokens"] * (fwd + bwd), "flops": 60 * D * c["tokens"]}
    lens = _lengths(c)
    T = int(lens.sum())
    if c["path"] == "delta":
        H, D, es = c["heads"], c["dim"], 1 if c["dtype"] == "e4m3" else 2
        rows = len(lens) * c["rows"]
        return {"bytes": 2 * (2 * T * H * D * es) + 4 * T * H * D + rows * H * D * (2 * es + 6),
                "flops": 14 * D * H * T * c["rows"]}
    if c["path"] == "layer":
        es = 1 if c["dtype"] == "e4m3" else 2
        nbytes = T * WIDTH * 2 * 4 + 3 * (2048 + 1536) * WIDTH * 2 + T * WIDTH * (3 * es + 2)
        return {"bytes": nbytes, "flops": 6 * T * WIDTH * (2048 + 1536) + 14 * WIDTH * _pairs(lens)}
    nbytes, flops = _attention_work(c, lens)
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    # about four times what each path measures against exact()
    if c["path"] == "gemm":
        return {"rel": 6e-3, "max": 0.1}    # one bf16 rounding of 32-bit sums: 1.7e-3
    if c["path"] == "norm":
        return {"rel": 6e-3, "max": 0.13}   # bf16 outputs 1.7e-3; an e4m3 value may round the other way
    if c["path"] == "delta":
        return {"rel": 1e-2, "max": 0.3}    # bf16 weights and outputs: 3.4e-3
    if c["path"] == "layer":
        # a rounding that changes travels through six stages: 2.7e-3 to 5.5e-3 in bf16; in FP8 a gradient
        # element may take the other of two e5m2 values, up to 25% apart (1e-1 against exact())
        return {"rel": 3e-2 if c["dtype"] == "e4m3" else 2e-2, "max": 0.8}
    return {"rel": 1e-2, "max": 0.4}        # 16-bit (or e4m3) weights between two products: 2.3e-3 in bf16


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, device="cuda", generator=g) * std).to(dtype)


def _offsets(lens):
    return torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device="cuda")


def _quantize(x):
    """e4m3 with one fp32 scale per row of the last axis."""
    s = (x.abs().amax(-1) / 448.0).float().clamp_min(1e-12)
    return (x / s[..., None]).to(E4M3), s


def _attention_inputs(c, seed):
    g, lens = _gen(seed), _lengths(c)
    T, H, D = int(lens.sum()), c["heads"], c["dim"]
    nt, window, prefix = _mask_options(c, lens)
    st = dict(N=c["max_len"], alpha=1.0 / D ** 0.5, offsets=_offsets(lens), window=window, prefix=prefix,
              nt=None if nt is None else torch.as_tensor(nt, device="cuda"), bias=None)
    if c["dtype"] == "e4m3":
        for name in ("q", "k", "v"):
            st[name], st[name + "s"] = _quantize(torch.randn(T, H, D, device="cuda", generator=g))
    else:
        for name in ("q", "k", "v"):
            st[name] = _randn(g, T, H, D, std=0.3)
    if c["mask"] == "bias":
        st["bias"] = _randn(g, H, 2 * _bias_span(c) - 1, std=0.02, dtype=torch.float32)
    if c["train"]:
        st["dout"] = _randn(g, T, H, D)
    return st


def _delta_inputs(c, seed):
    g, lens = _gen(seed), _lengths(c)
    T, B, H, D = int(lens.sum()), len(lens), c["heads"], c["dim"]
    st = dict(N=c["max_len"], alpha=1.0 / D ** 0.5, offsets=_offsets(lens))
    for name, rows in (("q", B * c["rows"]), ("k", T), ("v", T)):
        x = _randn(g, rows, H, D, std=0.5)
        st[name + "s"] = 1.0
        if c["dtype"] == "e4m3":
            st[name + "s"] = 0.008  # the calibrated per-tensor scale: about amax / 448 with headroom
            x = (x.float() / 0.008).clamp(-448, 448).to(E4M3)
        st[name] = x
    st["dout"] = _randn(g, B * c["rows"], H, D)
    return st


def _gemm_inputs(c, seed):
    g = _gen(seed)
    a8, a_scale = _quantize(torch.randn(c["m"], c["k"], device="cuda", generator=g))
    w8, w_scale = _quantize(torch.randn(c["n"], c["k"], device="cuda", generator=g) / c["k"] ** 0.5)
    return dict(a8=a8, a_scale=a_scale, weight=(w8, w_scale),
                bias=None if c["residual"] else _randn(g, c["n"], std=0.1),
                residual=_randn(g, c["m"], c["n"]) if c["residual"] else None,
                silu=(0, c["silu"]) if c["silu"] else None)


def _norm_inputs(c, seed):
    g, T = _gen(seed), c["tokens"]
    return dict(x=_randn(g, T, WIDTH), u=_randn(g, T, WIDTH), weight=1 + _randn(g, WIDTH, std=0.1),
                bias=_randn(g, WIDTH, std=0.05), dy=_randn(g, T, 3 * WIDTH))


def _layer_inputs(c, seed):
    g, lens = _gen(seed), _lengths(c)
    T = int(lens.sum())
    p = dict(input_norm_weight=1 + _randn(g, WIDTH, std=0.1), input_norm_bias=_randn(g, WIDTH, std=0.05),
             uvqk_weight=_randn(g, WIDTH, 2048, std=WIDTH ** -0.5), uvqk_bias=_randn(g, 2048, std=0.02),
             output_norm_weight=1 + _randn(g, WIDTH, std=0.1), output_norm_bias=_randn(g, WIDTH, std=0.05),
             output_weight=_randn(g, 1536, WIDTH, std=1536 ** -0.5))
    return dict(N=c["max_len"], offsets=_offsets(lens), x=_randn(g, T, WIDTH), dy=_randn(g, T, WIDTH),
                attn_bias=_randn(g, 4, 2 * _bias_span(c) - 1, std=0.02, dtype=torch.float32), params=p)


_INPUTS = dict(attention=_attention_inputs, delta=_delta_inputs, gemm=_gemm_inputs, norm=_norm_inputs,
               layer=_layer_inputs)


def prepare(c, seed):
    st = _INPUTS[c["path"]](c, seed)
    st["path"] = c["path"]
    if c["path"] == "attention" and c["train"]:
        st["grads"] = [torch.empty(st["q"].shape, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
        st["dbias"] = None if st["bias"] is None else torch.empty_like(st["bias"])
    if c["path"] == "delta":
        st["grads"] = [torch.empty(st[n].shape, dtype=torch.bfloat16, device="cuda") for n in ("q", "k", "v")]
    if c["path"] == "layer":
        for t in (st["x"], st["attn_bias"], *st["params"].values()):
            t.requires_grad_(True)
        st["options"] = {}
        if c["dtype"] == "e4m3":
            scale = lambda amax: torch.full((1,), amax * 1.5 / 448, device="cuda")  # noqa: E731
            st["options"] = dict(
                fp8_input_scale=scale(6.0), fp8_qkv_scale=scale(6.0), fp8_output_scale=scale(8.0),
                fp8_backward=bwd_fp8.Fp8BackwardConfig(
                    enabled=True, uvqk=True, out_wgrad_fp8=True, uvqk_wgrad_fp8t=True, outproj_lnmd_fused=True,
                    attn_full_fp8=True, warmup_calls=1, refresh_calls=1))
            for _ in range(3):  # the gradient scales settle, as they have in a running job
                run(st)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _run_attention(st):
    e4m3 = st["q"].dtype == E4M3
    scales = [st[n + "s"] for n in ("q", "k", "v")] if e4m3 else [None] * 3
    out = hstu_amd.triton_hstu_attention_fwd(
        st["N"], st["alpha"], st["q"], st["k"], st["v"], st["offsets"], st["nt"], st["window"], st["prefix"], None,
        False, 0, *scales, attn_bias=st["bias"])
    if "dout" not in st:
        return out
    dq, dk, dv = st["grads"]
    hstu_amd.triton_hstu_attention_bwd(
        st["dout"], st["q"], st["k"], st["v"], dq, dk, dv, st["offsets"], st["nt"], st["N"], st["alpha"],
        st["window"], st["prefix"], None, False, 0, *scales, attn_bias=st["bias"], dbias=st["dbias"])
    return out, dq, dk, dv, st["dbias"]


def _run_delta(st):
    dq, dk, dv = st["grads"]
    out = hstu_amd.triton_cached_hstu_mha(st["N"], st["alpha"], st["q"], st["k"], st["v"], st["offsets"],
                                          q_scale=st["qs"], k_scale=st["ks"], v_scale=st["vs"])
    hstu_amd.triton_hstu_attention_delta_bwd(st["dout"], st["q"], st["k"], st["v"], dq, dk, dv, st["offsets"],
                                             st["N"], st["alpha"], st["ks"], st["vs"], q_scale=st["qs"])
    return out, dq, dk, dv


def _run_gemm(st):
    return fp8.fp8_gemm(st["a8"], st["a_scale"], st["weight"], bias=st["bias"], residual=st["residual"],
                        silu_cols=st["silu"])


def _run_norm(st):
    y, mean, rstd, block_d, warps, seed, mask = hstu_amd.triton_layer_norm_mul_dropout_fwd(
        st["x"], st["u"], st["weight"], st["bias"], EPS, DROPOUT, True, True, True, True, "silu", DROPOUT_SEED,
        output_fp8=True, inv_scale=50.0)
    dx, du, dw, db, y16 = hstu_amd.triton_layer_norm_mul_dropout_bwd(
        st["dy"], st["x"], st["u"], st["weight"], st["bias"], mean, rstd, block_d, warps, EPS, True, DROPOUT, seed,
        True, True, True, "silu", compute_y=True, random_mask=mask)
    return y, mask, mean, rstd, dx, du, dw, db, y16


def _run_layer(st):
    leaves = [st["x"], st["attn_bias"], *st["params"].values()]
    for t in leaves:
        t.grad = None
    out = hstu_amd.hstu_layer(st["x"], st["offsets"], st["N"], st["params"], dropout_ratio=DROPOUT, training=True,
                              attn_bias=st["attn_bias"], seed=DROPOUT_SEED, norm_eps=EPS, **st["options"])
    out.backward(st["dy"])
    return [out.detach()] + [t.grad for t in leaves]


_RUN = dict(attention=_run_attention, delta=_run_delta, gemm=_run_gemm, norm=_run_norm, layer=_run_layer)


def run(st):
    return _RUN[st["path"]](st)


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _dense_bias(bias, length):
    span = (bias.shape[1] + 1) // 2
    i = torch.arange(length, device=bias.device)
    return bias[:, (i[:, None] - i[None, :]).clamp(-(span - 1), span - 1) + span - 1]


def _diagonal_sums(d, span):
    """Sums of d [H, L, L] over i - j, clamped to +-(span - 1): [H, 2 span - 1]."""
    H, L, _ = d.shape
    wide = torch.nn.functional.pad(d.flip(2), (0, L)).reshape(H, -1)[:, : L * (2 * L - 1)]
    sums = wide.reshape(H, L, 2 * L - 1).sum(1)  # column i - j + L - 1
    at = (torch.arange(2 * L - 1, device=d.device) - (L - 1)).clamp(-(span - 1), span - 1) + span - 1
    return torch.zeros(H, 2 * span - 1, dtype=d.dtype, device=d.device).index_add_(1, at, sums)


class _Attention(torch.autograd.Function):
    """silu(alpha q k^T + bias) / N, masked, times v, one sequence at a time."""

    @staticmethod
    def forward(ctx, q, k, v, bias, lens, N, alpha, masks):
        ctx.save_for_backward(q, k, v, bias)
        ctx.rest = lens, N, alpha, masks
        out, at = torch.empty_like(v), 0
        for b, L in enumerate(lens):
            s = _Attention.scores(q, k, bias, at, L, alpha)
            p = torch.nn.functional.silu(s) * _valid(L, *masks(b), q.device) / N
            out[at:at + L] = (p @ v[at:at + L].transpose(0, 1).contiguous()).transpose(0, 1)
            at += L
        return out

    @staticmethod
    def scores(q, k, bias, at, L, alpha):
        qh, kh = (x[at:at + L].transpose(0, 1).contiguous() for x in (q, k))
        s = qh @ kh.transpose(1, 2).contiguous() * alpha
        return s if bias is None else s + _dense_bias(bias, L)

    @staticmethod
    def backward(ctx, do):
        q, k, v, bias = ctx.saved_tensors
        lens, N, alpha, masks = ctx.rest
        dq, dk, dv, at = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), 0
        dbias = None if bias is None else torch.zeros_like(bias)
        for b, L in enumerate(lens):
            s = _Attention.scores(q, k, bias, at, L, alpha)
            sig = torch.sigmoid(s)
            valid = _valid(L, *masks(b), q.device) / N
            qh, kh, vh, doh = (x[at:at + L].transpose(0, 1).contiguous() for x in (q, k, v, do))
            dv[at:at + L] = ((s * sig * valid).transpose(1, 2).contiguous() @ doh).transpose(0, 1)
            ds = doh @ vh.transpose(1, 2).contiguous() * (sig * (1 + s * (1 - sig)) * valid)
            dq[at:at + L] = (ds @ kh).transpose(0, 1) * alpha
            dk[at:at + L] = (ds.transpose(1, 2).contiguous() @ qh).transpose(0, 1) * alpha
            if bias is not None:
                dbias += _diagonal_sums(ds, (bias.shape[1] + 1) // 2)
            at += L
        return dq, dk, dv, dbias, None, None, None, None


def _wide(x, scale=None):
    return x.double() if scale is None else x.double() * scale.double()[..., None]


def _exact_attention(c, seed):
    st, lens = _attention_inputs(c, seed), _lengths(c)
    nt, window, prefix = _mask_options(c, lens)
    q, k, v = (_wide(st[n], st.get(n + "s")).requires_grad_(c["train"]) for n in ("q", "k", "v"))
    bias = None if st["bias"] is None else st["bias"].double().requires_grad_(c["train"])
    out = _Attention.apply(q, k, v, bias, lens.tolist(), st["N"], st["alpha"],
                           lambda b: (None if nt is None else int(nt[b]), window, prefix))
    if not c["train"]:
        return out
    out.backward(st["dout"].double())
    return out.detach(), q.grad, k.grad, v.grad, None if bias is None else bias.grad


def _exact_delta(c, seed):
    st, lens, rows = _delta_inputs(c, seed), _lengths(c), c["rows"]
    q, k, v, do = (st[n].double() * st.get(n + "s", 1.0) for n in ("q", "k", "v", "dout"))
    out, dq, dk, dv, at = torch.empty_like(q), torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), 0
    for b, L in enumerate(lens.tolist()):
        r, t = slice(b * rows, (b + 1) * rows), slice(at, at + L)
        qh, kh, vh, doh = (x.transpose(0, 1).contiguous() for x in (q[r], k[t], v[t], do[r]))
        s = qh @ kh.transpose(1, 2).contiguous() * st["alpha"]
        valid = _valid(L, None, 0, 0, q.device)[L - rows:] / st["N"]
        sig = torch.sigmoid(s)
        p = s * sig * valid
        ds = doh @ vh.transpose(1, 2).contiguous() * (sig * (1 + s * (1 - sig)) * valid)
        out[r] = (p @ vh).transpose(0, 1)
        dq[r] = (ds @ kh).transpose(0, 1) * st["alpha"]
        dk[t] = (ds.transpose(1, 2).contiguous() @ qh).transpose(0, 1) * st["alpha"]
        dv[t] = (p.transpose(1, 2).contiguous() @ doh).transpose(0, 1)
        at += L
    return out, dq, dk, dv


def _exact_gemm(c, seed):
    st = _gemm_inputs(c, seed)
    out = _wide(st["a8"], st["a_scale"]) @ _wide(*st["weight"]).t().contiguous()
    if st["bias"] is not None:
        out += st["bias"].double()
    if st["silu"] is not None:
        out[:, : c["silu"]] = torch.nn.functional.silu(out[:, : c["silu"]])
    return out if st["residual"] is None else out + st["residual"].double()


def _keep_bits(T):
    """The 16-bit dropout masks [T, D]: Philox4x32-10 on one counter per eight
    rows, mask and column; bit 0 keeps y, bit 1 x, bit 2 u."""
    low32 = 0xFFFFFFFF
    groups = (T + 7) // 8
    threshold = round(DROPOUT * 65536)
    keep = torch.zeros(groups, 8, WIDTH, dtype=torch.int8, device="cuda")
    g = torch.arange(groups, device="cuda")[:, None] * (3 * WIDTH)
    col = torch.arange(WIDTH, device="cuda")[None, :]
    for j in range(3):
        c0 = (g + j * WIDTH + col) & low32
        c1, c2, c3 = (torch.zeros_like(c0) for _ in range(3))
        ka, kb = DROPOUT_SEED & low32, DROPOUT_SEED >> 32
        for _ in range(10):
            pa, pb = c0 * 0xD2511F53, c2 * 0xCD9E8D57  # 64-bit products, modulo 2^64
            c0, c1, c2, c3 = ((pb >> 32) & low32) ^ c1 ^ ka, pb & low32, ((pa >> 32) & low32) ^ c3 ^ kb, pa & low32
            ka, kb = (ka + 0x9E3779B9) & low32, (kb + 0xBB67AE85) & low32
        for i, word in enumerate((c0, c1, c2, c3)):
            keep[:, i] |= ((word & 0xFFFF) >= threshold).to(torch.int8) << j
            keep[:, i + 4] |= ((word >> 16) >= threshold).to(torch.int8) << j
    return keep.reshape(-1, WIDTH)[:T]


def _norm_mul_dropout(x, u, weight, bias, keep):
    y = torch.nn.functional.layer_norm(x, (WIDTH,), weight, bias, EPS) * torch.nn.functional.silu(u)
    blocks = (torch.nn.functional.silu(u), x, y)
    return torch.cat([b * ((keep >> bit) & 1) / (1 - DROPOUT) for b, bit in zip(blocks, (2, 1, 0))], 1)


def _exact_norm(c, seed):
    st = _norm_inputs(c, seed)
    keep = _keep_bits(c["tokens"])
    x, u, w, b = (st[n].double().requires_grad_(True) for n in ("x", "u", "weight", "bias"))
    y = _norm_mul_dropout(x, u, w, b, keep)
    y.backward(st["dy"].double())
    y, xd = y.detach(), x.detach()
    rstd = 1 / torch.sqrt(xd.var(1, unbiased=False) + EPS)
    return (y * 50.0).clamp(-448, 448), None, xd.mean(1), rstd, x.grad, u.grad, w.grad, b.grad, y


def _exact_layer(c, seed):
    st, lens = _layer_inputs(c, seed), _lengths(c)
    T = int(lens.sum())
    leaves = [t.double().requires_grad_(True) for t in (st["x"], st["attn_bias"], *st["params"].values())]
    x, attn_bias = leaves[:2]
    p = dict(zip(st["params"], leaves[2:]))
    xn = torch.nn.functional.layer_norm(x, (WIDTH,), p["input_norm_weight"], p["input_norm_bias"], EPS)
    u, v, q, k = torch.split(xn @ p["uvqk_weight"] + p["uvqk_bias"], WIDTH, dim=1)
    q, k, v = (t.reshape(T, 4, 128) for t in (q, k, v))
    attn = _Attention.apply(q, k, v, attn_bias, lens.tolist(), st["N"], 128 ** -0.5, lambda b: (None, 0, 0))
    y = _norm_mul_dropout(attn.reshape(T, WIDTH), u, p["output_norm_weight"], p["output_norm_bias"], _keep_bits(T))
    out = y @ p["output_weight"] + x
    out.backward(st["dy"].double())
    # the FP8 weight gradients are sums of e5m2 values (two mantissa bits): 64 bits say little about them
    return [out.detach(), x.grad] + [None if c["dtype"] == "e4m3" else t.grad for t in leaves[1:]]


_EXACT = dict(attention=_exact_attention, delta=_exact_delta, gemm=_exact_gemm, norm=_exact_norm, layer=_exact_layer)


def exact(c, seed):
    return _EXACT[c["path"]](c, seed)
