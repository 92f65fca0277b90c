"""The work whose speed counts: what a user's program has this library do, case by case.

Each case is one pass through the public functions (rmsnorm, geglu, geglu_linear,
relpos_attention, t5_relpos_table), as a layer of a model calls them: a forward without
gradients in inference, a forward and its backward in training. `listed()` has the named
cases, `draw()` further ones of the same ranges.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

# The working folder is the root of the tree whose library is used.
_LIBRARY = str(Path("kernel-rsi_amd/library").resolve())
if _LIBRARY not in sys.path:
    sys.path.insert(0, _LIBRARY)
import geglu as geglu_mod  # noqa: E402
import relpos_attention as attn_mod  # noqa: E402
import rmsnorm as rmsnorm_mod  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EPS = 1e-6


def listed() -> list[dict]:
    return [
        # One norm of one short ragged sequence at inference: the smallest call there is.
        {"name": "rmsnorm_infer_300x1152_bf16", "op": "rmsnorm", "train": False, "dtype": "bf16",
         "rows": 300, "n": 1152},
        # The norm of a mid-sized training layer, with a row count no tile divides.
        {"name": "rmsnorm_train_8191x1152_bf16", "op": "rmsnorm", "train": True, "dtype": "bf16",
         "rows": 8191, "n": 1152},
        # The norm of a large training layer, batch 8 x 4096 tokens of width 4096.
        {"name": "rmsnorm_train_32768x4096_bf16", "op": "rmsnorm", "train": True, "dtype": "bf16",
         "rows": 32768, "n": 4096},
        # A gated MLP of two thirds of 4 x 1024 columns, in fp16: neither the width nor the row
        # count is a multiple of a vector load.
        {"name": "geglu_train_4099x2730_tanh_fp16", "op": "geglu", "train": True, "dtype": "fp16",
         "rows": 4099, "f": 2730, "approximate": "tanh"},
        # The gated MLP activation of a large training layer, exact GELU.
        {"name": "geglu_train_8192x4096_erf_bf16", "op": "geglu", "train": True, "dtype": "bf16",
         "rows": 8192, "f": 4096, "approximate": "none"},
        # The merged projection with its activation at inference (prefill of 8192 tokens).
        {"name": "geglu_linear_infer_8192x4096x4096_bf16", "op": "geglu_linear", "train": False,
         "dtype": "bf16", "rows": 8192, "k": 4096, "f": 4096, "approximate": "tanh"},
        # The same layer of a smaller model in training, over a ragged batch of tokens.
        {"name": "geglu_linear_train_1000x1024x2816_bf16", "op": "geglu_linear", "train": True,
         "dtype": "bf16", "rows": 1000, "k": 1024, "f": 2816, "approximate": "tanh"},
        # Attention of an encoder or diffusion block at inference, head dim 72.
        {"name": "attn_infer_b2_s1024_h16_d72_bf16", "op": "attention", "train": False, "dtype": "bf16",
         "b": 2, "s": 1024, "h": 16, "d": 72, "t5": False},
        # One T5 encoder layer's attention in training: the bias comes from the bucket table.
        {"name": "attn_train_t5_b4_s512_h16_d64_bf16", "op": "attention", "train": True, "dtype": "bf16",
         "b": 4, "s": 512, "h": 16, "d": 64, "t5": True},
        # Attention in fp16 training over a ragged length.
        {"name": "attn_train_b3_s1021_h12_d80_fp16", "op": "attention", "train": True, "dtype": "fp16",
         "b": 3, "s": 1021, "h": 12, "d": 80, "t5": False},
        # Attention in full fp32 training (no reduced-precision products anywhere).
        {"name": "attn_train_b2_s1024_h16_d72_fp32", "op": "attention", "train": True, "dtype": "fp32",
         "b": 2, "s": 1024, "h": 16, "d": 72, "t5": False},
        # Attention of a large training layer over long sequences.
        {"name": "attn_train_b4_s4096_h16_d64_bf16", "op": "attention", "train": True, "dtype": "bf16",
         "b": 4, "s": 4096, "h": 16, "d": 64, "t5": False},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo: int, hi: int) -> int:
    """A width: mostly a multiple of 8, one in four as it falls."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.25 else max(lo, n // 8 * 8)


def draw(rng) -> dict:
    op = rng.choice(["rmsnorm", "geglu", "geglu_linear", "attention", "attention"])
    train = rng.random() < 0.7
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if op == "rmsnorm":
        return {"op": op, "train": train, "dtype": dtype, "rows": _log_int(rng, 64, 16384),
                "n": _width(rng, 256, 8192)}
    approximate = rng.choice(["tanh", "none"])
    if op == "geglu":
        return {"op": op, "train": train, "dtype": dtype, "rows": _log_int(rng, 64, 8192),
                "f": _width(rng, 256, 8192), "approximate": approximate}
    if op == "geglu_linear":
        rows, k = _log_int(rng, 64, 4096 if train else 8192), _log_int(rng, 4, 64) * 64
        f = _log_int(rng, 4, 64) * 64
        return {"op": op, "train": train, "dtype": rng.choice(["bf16", "fp16"]), "rows": rows, "k": k, "f": f,
                "approximate": approximate}
    d = rng.choice([32, 40, 64, 64, 64, 72, 80, 96, 128])
    s = _log_int(rng, 64, 2048 if dtype == "fp32" else 4096)
    # b h s^2 d is bounded so that no drawn case takes longer than the largest listed one (fp32
    # products run at a sixteenth of the 16-bit rate).
    budget = (1 << 31) if dtype == "fp32" else (3 << 34)
    bh_max = max(4, min(64, budget // (s * s * d)))
    h = min(_log_int(rng, 2, 16), bh_max)
    b = max(1, min(_log_int(rng, 1, 8), bh_max // h))
    return {"op": op, "train": train, "dtype": dtype, "b": b, "s": s, "h": h, "d": d,
            "t5": rng.random() < 0.3}


# ------------------------------------------------------------------ one case
def _randn(gen, shape, dtype, std=1.0, mean=0.0):
    t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return t.mul_(std).add_(mean).to(dtype)


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt, train = DTYPES[case["dtype"]], case["train"]
    st = {"case": case}
    if case["op"] == "rmsnorm":
        st["x"] = _randn(gen, (case["rows"], case["n"]), dt)
        st["w"] = _randn(gen, (case["n"],), dt, std=0.1, mean=1.0)
        grad_shape, leaves = st["x"].shape, ("x", "w")
    elif case["op"] == "geglu":
        st["u"] = _randn(gen, (case["rows"], 2 * case["f"]), dt)
        grad_shape, leaves = (case["rows"], case["f"]), ("u",)
    elif case["op"] == "geglu_linear":
        st["x"] = _randn(gen, (case["rows"], case["k"]), dt)
        st["w"] = _randn(gen, (2 * case["f"], case["k"]), dt, std=case["k"] ** -0.5)
        grad_shape, leaves = (case["rows"], case["f"]), ("x", "w")
    else:
        b, s, h, d = (case[k] for k in "bshd")
        st["qkv"] = _randn(gen, (b * s, 3 * h * d), dt)
        if case["t5"]:
            st["table"] = _randn(gen, (32, h), torch.float32, std=0.5)
        else:
            st["pd"] = _randn(gen, (h, 2 * s - 1), torch.float32, std=0.5)
        grad_shape, leaves = (b * s, h * d), ("qkv", "table" if case["t5"] else "pd")
    if train:
        st["dout"] = _randn(gen, grad_shape, dt)
        st["leaves"] = [st[k].requires_grad_(True) for k in leaves]
    return st


def _forward(st: dict):
    case = st["case"]
    if case["op"] == "rmsnorm":
        return rmsnorm_mod.rmsnorm(st["x"], st["w"], EPS)
    if case["op"] == "geglu":
        return geglu_mod.geglu(st["u"], approximate=case["approximate"])
    if case["op"] == "geglu_linear":
        return geglu_mod.geglu_linear(st["x"], st["w"], approximate=case["approximate"])
    b, s, h, d = (case[k] for k in "bshd")
    pd = attn_mod.t5_relpos_table(st["table"], s) if case["t5"] else st["pd"]
    return attn_mod.relpos_attention(st["qkv"], pd, b, s, h, d, d ** -0.5)


def run(st: dict) -> dict:
    if not st["case"]["train"]:
        with torch.no_grad():
            return {"out": _forward(st)}
    out = _forward(st)
    grads = torch.autograd.grad(out, st["leaves"], st["dout"])
    return {"out": out.detach(), "grads": list(grads)}


# ---------------------------------------------------------------- what counts
def work(case: dict) -> dict:
    e = DTYPES[case["dtype"]].itemsize
    train = case["train"]
    if case["op"] == "rmsnorm":
        m = case["rows"] * case["n"]
        # x -> y; and x, dy -> dx, with w and dw.
        nbytes = e * (2 * m + case["n"]) + (e * (3 * m + 2 * case["n"]) if train else 0)
        return {"bytes": nbytes, "flops": m * (4 + (12 if train else 0))}
    if case["op"] == "geglu":
        m = case["rows"] * case["f"]
        return {"bytes": e * m * (3 + (5 if train else 0)), "flops": m * (12 + (25 if train else 0))}
    if case["op"] == "geglu_linear":
        r, k, f = case["rows"], case["k"], case["f"]
        nbytes = e * (r * k + 2 * f * k + r * f) + (e * (r * f + 2 * (r * k + 2 * f * k)) if train else 0)
        return {"bytes": nbytes, "flops": 4 * r * k * f * (3 if train else 1)}
    b, s, h, d = (case[k] for k in "bshd")
    tok = b * s * h * d
    nbytes = e * 4 * tok + 4 * h * (2 * s - 1)
    if train:
        nbytes += e * (3 + 1 + 3) * tok + 8 * h * (2 * s - 1)
    return {"bytes": nbytes, "flops": b * h * s * s * d * (14 if train else 4)}


def tolerance(case: dict) -> dict:
    """About four times the 2-norm error against 64 bits measured over these ranges: bf16
    0.0023-0.0035, fp16 0.00028-0.00045, fp32 up to 8e-7 in attention (growing with the length)
    and 1.6e-7 elsewhere."""
    if case["dtype"] == "fp32":
        return {"rel": 5e-6 if case["op"] == "attention" else 1e-6}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}


# ------------------------------------------------------------------ in 64 bits
def exact(case: dict, seed: int):
    st = prepare(case, seed)
    if case["op"] == "attention":
        return _exact_attention(st)
    f64 = {k: st[k].detach().double() for k in ("x", "w", "u") if k in st}
    if case["train"]:
        for t in f64.values():
            t.requires_grad_(True)
    if case["op"] == "rmsnorm":
        x, w = f64["x"], f64["w"]
        out = w * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS))
        leaves = [x, w] if case["train"] else None
    else:
        u = f64["u"] if case["op"] == "geglu" else f64["x"] @ f64["w"].t()
        a, b = u.chunk(2, dim=-1)
        out = torch.nn.functional.gelu(a, approximate=case["approximate"]) * b
        leaves = [f64["u"]] if case["op"] == "geglu" else [f64["x"], f64["w"]]
    if not case["train"]:
        return {"out": out}
    grads = torch.autograd.grad(out, leaves, st["dout"].double())
    return {"out": out.detach(), "grads": list(grads)}


def _t5_bucket(s: int) -> torch.Tensor:
    """T5's bidirectional bucket (32 buckets, distances up to 128) of j - i = r - (s - 1)."""
    dist = torch.arange(2 * s - 1, device="cuda") - (s - 1)
    a = dist.abs()
    large = 8 + (torch.log(a.float() / 8) / math.log(128 / 8) * 8).long()
    return (dist > 0).long() * 16 + torch.where(a < 8, a, large.clamp(max=15))


@torch.no_grad()
def _exact_attention(st: dict):
    case = st["case"]
    b, s, h, d = (case[k] for k in "bshd")
    scale = d ** -0.5
    qkv = st["qkv"].double().view(b, s, 3, h, d)
    bucket = _t5_bucket(s) if case["t5"] else None
    pd = st["table"].double()[bucket].t().contiguous() if case["t5"] else st["pd"].double()
    pos = torch.arange(s, device="cuda")
    r = pos[None, :] - pos[:, None] + s - 1
    out = torch.empty(b, s, h, d, device="cuda", dtype=torch.float64)
    if case["train"]:
        dout = st["dout"].double().view(b, s, h, d)
        dqkv, dpd = torch.empty_like(qkv), torch.zeros_like(pd)
    for hi in range(h):
        bias = pd[hi][r]
        for bi in range(b):
            q, k, v = (qkv[bi, :, i, hi].contiguous() for i in range(3))
            p = torch.softmax(q @ k.t() * scale + bias, dim=-1)
            o = p @ v
            out[bi, :, hi] = o
            if not case["train"]:
                continue
            do = dout[bi, :, hi].contiguous()
            ds = p * (do @ v.t() - (do * o).sum(-1, keepdim=True))
            dqkv[bi, :, 0, hi] = ds @ k * scale
            dqkv[bi, :, 1, hi] = ds.t() @ q * scale
            dqkv[bi, :, 2, hi] = p.t() @ do
            # Row i shifted right by s - 1 - i: column j - i + s - 1 then holds diagonal j - i.
            skew = torch.nn.functional.pad(ds.flip(0), (0, s)).flatten()[: s * (2 * s - 1)]
            dpd[hi] += skew.view(s, 2 * s - 1).sum(0)
    out = out.view(b * s, h * d)
    if not case["train"]:
        return {"out": out}
    if case["t5"]:
        dpd = torch.zeros(32, h, device="cuda", dtype=torch.float64).index_add_(0, bucket, dpd.t().contiguous())
    return {"out": out, "grads": [dqkv.view(b * s, 3 * h * d), dpd]}
