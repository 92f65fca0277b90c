"""fp16 and fp32 activations (the reference's kernels are dtype-generic): the HIP kernels vs
the fp32 reference, with the eager original in the same dtype as the noise yardstick.

Tolerance, stated: the reference's acceptance criterion with slack 2 (tools/common.py:
322-392, 476-490), as for bf16: every output's max error and rel-L2 within 2x those of the
eager original in the same dtype, per-row errors within 3x, with the criterion's absolute
floors (1e-3 of the peak per element, 1e-5 rel-L2), which is what an fp32 run is held to.
Attention in fp16 is additionally held to the reference Triton kernels' own rounding points
(P and dS rounded to fp16), per row at 3x. Attention in fp32 (P and dS unrounded as
the reference keeps them for fp32 inputs) is held to the same criterion against a float64
reference of the same fp32 inputs, with the eager fp32 computation as the yardstick; in practice
that is the floors (1e-5 rel-L2, 1e-3 of the peak per element, per-row 3x the median row error
+ 1e-5), far tighter than the reference's own fp32 path, which runs its products in TF32.
"""
import math

import pytest
import torch

import _hip
import geglu as G
import krsi_oracle as O
import relpos_attention as A
import rmsnorm as R
from krsi_testutil import assert_parity, log, seeded

pytestmark = pytest.mark.gpu
EPS = 1e-6
DTYPES = [torch.float16, torch.float32]


def _name(dt):
    return str(dt).replace("torch.", "")


# ------------------------------------------------------------------- RMSNorm
def _rms(x, w, g, dt):
    ref32 = O.rmsnorm_train(x, w, EPS, g.float(), torch.float32)
    orig = O.rmsnorm_train(x, w, EPS, g, dt)
    xx = x.detach().requires_grad_(True)
    ww = w.detach().requires_grad_(True)
    y = R.rmsnorm(xx, ww, EPS)
    dx, dw = torch.autograd.grad(y, [xx, ww], g)
    assert y.dtype == dt and dx.dtype == dt and dw.dtype == dt
    return ref32, orig, (y.detach(), dx, dw)


@pytest.mark.parametrize("dt", DTYPES, ids=_name)
@pytest.mark.parametrize("rows,n", [(2048, 1152), (300, 4096), (5, 7), (33, 1001), (64, 256),
                                    (9, 8192), (5, 16384), (1000, 512)])
def test_rmsnorm_dtypes(dt, rows, n):
    log(f"rmsnorm {_name(dt)} rows={rows} n={n}")
    x = seeded((rows, n), 30 + n, dtype=dt)
    w = seeded((n,), 31, std=0.1, mean=1.0, dtype=dt)
    g = seeded((rows, n), 32, dtype=dt)
    ref32, orig, cand = _rms(x, w, g, dt)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand, extra_msg=_name(dt))
    # The forward against the eager original of the same dtype: in fp16 bitwise except at
    # rounding ties of x*r (fp32 statistics summed in another order); in fp32, which has no
    # rounding point to absorb that order, within a few fp32 ulps.
    eager = O.rmsnorm(x, w, EPS)
    if dt == torch.float16:
        same = (cand[0] == eager).float().mean().item()
        assert same > 0.999, same
    else:
        assert torch.allclose(cand[0], eager, rtol=4e-7 * 8, atol=1e-7), (cand[0] - eager).abs().max()


@pytest.mark.parametrize("dt", DTYPES, ids=_name)
def test_rmsnorm_dtypes_unaligned_and_deterministic(dt):
    log(f"rmsnorm {_name(dt)} unaligned view + determinism")
    base = seeded((64 * 256 + 1,), 33, dtype=dt)
    x = base[1:].view(64, 256)
    w = seeded((256,), 34, std=0.1, mean=1.0, dtype=dt)
    g = seeded((64, 256), 35, dtype=dt)
    ref32, orig, cand = _rms(x, w, g, dt)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand, extra_msg=_name(dt))
    x = seeded((2048, 4096), 36, dtype=dt)
    w = seeded((4096,), 37, std=0.02, mean=1.0, dtype=dt)
    g = seeded((2048, 4096), 38, dtype=dt)
    _, rstd = _hip.rmsnorm_fwd(x, w, EPS)
    a = _hip.rmsnorm_bwd(g, x, w, rstd)
    b = _hip.rmsnorm_bwd(g, x, w, rstd)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_rmsnorm_mixed_dtypes_rejected():
    x = seeded((4, 64), 1, dtype=torch.float16)
    with pytest.raises(TypeError):
        R.rmsnorm(x, torch.ones(64, device="cuda", dtype=torch.float32), EPS)
    with pytest.raises(TypeError):
        R.rmsnorm(x.double(), torch.ones(64, device="cuda", dtype=torch.float64), EPS)


# --------------------------------------------------------------------- GEGLU
@pytest.mark.parametrize("dt", DTYPES, ids=_name)
@pytest.mark.parametrize("approximate", ["none", "tanh"])
@pytest.mark.parametrize("rows,f", [(1, 8), (7, 1001), (64, 2816), (300, 64), (2, 4100), (512, 4096)])
def test_geglu_dtypes(dt, approximate, rows, f):
    log(f"geglu {_name(dt)} {approximate} rows={rows} f={f}")
    u = seeded((rows, 2 * f), 40 + f, std=2.0, dtype=dt)
    g = seeded((rows, f), 41, dtype=dt)
    ref32 = O.geglu_train(u, g.float(), approximate, torch.float32)
    orig = O.geglu_train(u, g, approximate, dt)
    uu = u.detach().requires_grad_(True)
    out = G.geglu(uu, approximate=approximate)
    (du,) = torch.autograd.grad(out, [uu], g)
    assert out.dtype == dt and du.dtype == dt
    assert_parity(["out", "du"], ref32, orig, (out.detach(), du), extra_msg=_name(dt))


# ------------------------------------------------ relative-position attention
def _relpos_fp16(B, S, H, D, scale, std=1.0, pd_std=0.02, ref_device="cpu", ld_extra=0, seed=50,
                 pd_fn=None, vs_eager=True):
    dt = torch.float16
    qkv = seeded((B * S, 3 * H * D + ld_extra), seed, std=std, dtype=dt)
    if ld_extra:
        qkv = qkv[:, :3 * H * D]
    pd = seeded((H, 2 * S - 1), seed + 1, std=pd_std, dtype=torch.float32)
    if pd_fn is not None:
        pd = pd_fn(pd)
    dout = seeded((B * S, H * D), seed + 2, dtype=dt)
    x = qkv.detach().requires_grad_(True)
    p = pd.detach().requires_grad_(True)
    out = A.relpos_attention(x, p, B, S, H, D, scale)
    dqkv, dpd = torch.autograd.grad(out, [x, p], dout)
    assert out.dtype == dt and dqkv.dtype == dt and dpd.dtype == torch.float32
    dev = torch.device(ref_device)
    a = (qkv.to(dev), pd.to(dev), B, S, H, D, scale, dout.to(dev))
    r = O.relpos_manual(*a)
    o = O.relpos_manual(*a, eager_dtype=dt)
    kem = O.relpos_kernel_emulated(*a, dtype=dt)
    cand = (out.detach().to(dev), dqkv.to(dev), dpd.to(dev))
    tag = f"fp16 B{B} S{S} H{H} D{D}"
    if vs_eager:
        assert_parity(["out", "dqkv", "dpd"], (r[0], r[2], r[3]), (o[0], o[2], o[3]), cand,
                      row_slack=float("inf"), extra_msg=tag + " vs eager fp16")
    assert_parity(["out", "dqkv", "dpd"], (r[0], r[2], r[3]), kem, cand,
                  extra_msg=tag + " vs reference-kernel rounding")
    _, out32, lse = _hip.relpos_fwd(qkv, pd, B, S, H, D, scale)
    assert torch.allclose(lse.to(dev), r[1], atol=1e-3, rtol=1e-4)
    assert (out32.to(dev) - r[0]).norm() / r[0].norm() < 1e-3


FP16_CASES = [  # B, S, H, D, scale, qkv std, pd std
    (1, 2, 1, 64, 0.125, 1.0, 0.02),
    (1, 17, 2, 32, 0.2, 1.0, 1.0),
    (2, 64, 2, 64, 1.0, 0.6, 1.0),
    (1, 128, 2, 128, 1 / math.sqrt(128), 1.0, 0.02),
    (2, 300, 2, 72, 1 / math.sqrt(72), 1.0, 0.02),
    (1, 257, 1, 8, 0.35, 1.0, 0.3),
    (1, 96, 2, 64, -0.125, 1.0, 0.5),
    (1, 80, 2, 32, 0.0, 1.0, 1.0),
]


@pytest.mark.parametrize("B,S,H,D,scale,std,pd_std", FP16_CASES)
def test_relpos_fp16(B, S, H, D, scale, std, pd_std):
    log(f"relpos fp16 B{B} S{S} H{H} D{D} scale {scale:.4g}")
    _relpos_fp16(B, S, H, D, scale, std, pd_std)


def test_relpos_fp16_strided_and_large():
    log("relpos fp16 strided qkv B2 S96 H2 D64")
    _relpos_fp16(2, 96, 2, 64, 0.125, ld_extra=40)
    log("relpos fp16 B2 S1024 H16 D72")
    _relpos_fp16(2, 1024, 16, 72, 1 / math.sqrt(72), ref_device="cuda")
    # D 64 with 256 blocks of each backward kind: the one-launch dQ + dK/dV pairing.
    log("relpos fp16 B2 S1024 H16 D64")
    _relpos_fp16(2, 1024, 16, 64, 0.125, ref_device="cuda")


def _relpos_fp32(B, S, H, D, scale, std=1.0, pd_std=0.02, ref_device="cpu", ld_extra=0, seed=70,
                 pd_fn=None):
    dt = torch.float32
    qkv = seeded((B * S, 3 * H * D + ld_extra), seed, std=std, dtype=dt)
    if ld_extra:
        qkv = qkv[:, :3 * H * D]
    pd = seeded((H, 2 * S - 1), seed + 1, std=pd_std, dtype=torch.float32)
    if pd_fn is not None:
        pd = pd_fn(pd)
    dout = seeded((B * S, H * D), seed + 2, dtype=dt)
    x = qkv.detach().requires_grad_(True)
    p = pd.detach().requires_grad_(True)
    out = A.relpos_attention(x, p, B, S, H, D, scale)
    dqkv, dpd = torch.autograd.grad(out, [x, p], dout)
    assert out.dtype == dt and dqkv.dtype == dt and dpd.dtype == torch.float32
    dev = torch.device(ref_device)
    a = (qkv.to(dev), pd.to(dev), B, S, H, D, scale, dout.to(dev))
    r = O.relpos_manual(*a, compute_dtype=torch.float64)
    o = O.relpos_manual(*a)  # the eager fp32 computation (explicit fp32 matmuls + softmax)
    cand = (out.detach().to(dev), dqkv.to(dev), dpd.to(dev))
    tag = f"fp32 B{B} S{S} H{H} D{D}"
    assert_parity(["out", "dqkv", "dpd"], (r[0], r[2], r[3]), (o[0], o[2], o[3]), cand,
                  extra_msg=tag + " vs eager fp32")
    _, out32, lse = _hip.relpos_fwd(qkv, pd, B, S, H, D, scale)
    assert torch.equal(out32, out.detach())
    assert torch.allclose(lse.to(dev).double(), r[1], atol=1e-5, rtol=1e-6), (lse.to(dev) - r[1]).abs().max()


FP32_CASES = [  # B, S, H, D, scale, qkv std, pd std
    (1, 2, 1, 64, 0.125, 1.0, 0.02),
    (1, 17, 2, 32, 0.2, 1.0, 1.0),
    (2, 64, 2, 64, 1.0, 0.6, 1.0),
    (1, 128, 2, 128, 1 / math.sqrt(128), 1.0, 0.02),
    (2, 300, 2, 72, 1 / math.sqrt(72), 1.0, 0.02),
    (1, 200, 1, 16, 0.25, 1.0, 0.5),
    (1, 130, 2, 48, 0.3, 1.0, 0.02),
    (1, 100, 1, 80, 0.1, 1.0, 0.02),
    (1, 96, 2, 96, 0.1, 1.0, 0.02),
    (1, 70, 1, 112, 0.1, 1.0, 0.02),
    (1, 257, 1, 8, 0.35, 1.0, 0.3),
    (1, 96, 2, 64, -0.125, 1.0, 0.5),
    (1, 80, 2, 32, 0.0, 1.0, 1.0),
]


@pytest.mark.parametrize("B,S,H,D,scale,std,pd_std", FP32_CASES)
def test_relpos_fp32(B, S, H, D, scale, std, pd_std):
    log(f"relpos fp32 B{B} S{S} H{H} D{D} scale {scale:.4g}")
    _relpos_fp32(B, S, H, D, scale, std, pd_std)


def _mask(kind, S):
    """-inf entries of the table: keys after the query (causal) or more than 16 away (band16)."""
    def fn(pd):
        r = torch.arange(2 * S - 1, device=pd.device) - (S - 1)
        keep = r <= 0 if kind == "causal" else r.abs() <= 16
        return pd.masked_fill(~keep, float("-inf"))
    return fn


@pytest.mark.parametrize("mask", ["causal", "band16"])
def test_relpos_fp16_fp32_masks_through_the_bias(mask):
    """Masked relative positions in fp32 (against float64, with the eager fp32 yardstick) and
    fp16 (against the reference kernel's rounding points, as the bf16 masked cases). band16
    masks whole leading key steps of the later queries."""
    log(f"relpos fp32 {mask} mask B2 S160 H2 D64")
    _relpos_fp32(2, 160, 2, 64, 0.125, pd_std=0.5, pd_fn=_mask(mask, 160))
    log(f"relpos fp16 {mask} mask B2 S160 H2 D64")
    _relpos_fp16(2, 160, 2, 64, 0.125, pd_std=0.5, pd_fn=_mask(mask, 160), vs_eager=False)


def test_relpos_fp32_single_position():
    """S = 1: out = v and dv = dout exactly (p = 1 in both passes); dq, dk and dpd are 0 up to
    the rounding of dp - delta, whose two dot products are summed in different orders."""
    B, S, H, D = 2, 1, 3, 64
    qkv = seeded((B * S, 3 * H * D), 80, dtype=torch.float32)
    pd = seeded((H, 1), 81, dtype=torch.float32)
    dout = seeded((B * S, H * D), 82, dtype=torch.float32)
    x = qkv.detach().requires_grad_(True)
    p = pd.detach().requires_grad_(True)
    out = A.relpos_attention(x, p, B, S, H, D, 0.125)
    dqkv, dpd = torch.autograd.grad(out, [x, p], dout)
    q, k, v = O.split_qkv(qkv, B, S, H, D)
    assert torch.equal(out.detach(), v.permute(0, 2, 1, 3).reshape(B * S, H * D))
    d = dqkv.view(B * S, 3, H * D)
    assert torch.equal(d[:, 2], dout)
    assert d[:, :2].abs().max().item() < 1e-5 and dpd.abs().max().item() < 1e-5


def test_relpos_fp32_strided_and_config4_shape():
    """A qkv row stride wider than 3*H*D, then the BASELINE config 4 shape (B2 H16 L1024 D72)
    forward and backward against the float64 reference on the GPU; the backward is bitwise
    reproducible."""
    log("relpos fp32 strided qkv B2 S96 H2 D64")
    _relpos_fp32(2, 96, 2, 64, 0.125, ld_extra=40)
    log("relpos fp32 B2 S1024 H16 D72 (config 4 shape)")
    _relpos_fp32(2, 1024, 16, 72, 1 / math.sqrt(72), ref_device="cuda")
    B, S, H, D = 2, 1024, 16, 72
    qkv = seeded((B * S, 3 * H * D), 90, dtype=torch.float32)
    pd = seeded((H, 2 * S - 1), 91, std=0.02, dtype=torch.float32)
    dout = seeded((B * S, H * D), 92, dtype=torch.float32)
    _, out32, lse = _hip.relpos_fwd(qkv, pd, B, S, H, D, 0.1)
    a = _hip.relpos_bwd(dout, qkv, pd, out32, lse, B, S, H, D, 0.1)
    b = _hip.relpos_bwd(dout, qkv, pd, out32, lse, B, S, H, D, 0.1)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_relpos_fp16_config5_shape():
    """The BASELINE config 5 shape in fp16 (B4 H16 L4096 D64), against the fp32 reference on the
    GPU, with the same two criteria as the small cases."""
    log("relpos fp16 B4 S4096 H16 D64")
    _relpos_fp16(4, 4096, 16, 64, 1 / 8, ref_device="cuda")


@pytest.mark.parametrize("S", [8191, 16384])
def test_relpos_fp16_fp32_long_sequence(S):
    """Long context in fp16 and fp32 (B1 H2 D64), against the fp32 reference on the GPU: the odd
    S = 8191 takes the scalar dpd reduce, S = 16384 the 128-bit one, as in bf16."""
    log(f"relpos fp16 long context B1 S{S} H2 D64")
    _relpos_fp16(1, S, 2, 64, 0.125, ref_device="cuda")
    log(f"relpos fp32 long context B1 S{S} H2 D64")
    _relpos_fp32(1, S, 2, 64, 0.125, ref_device="cuda")


def test_relpos_fp32_non_finite_elements():
    """An infinite element has no exact bf16 parts: its workgroup redoes the tile with fp32
    products. One infinite v (forward) and one infinite dout (backward) in head 0: exactly the
    outputs that IEEE makes infinite or NaN are, the rest match the finite formulas in float64,
    and head 1 is bitwise that of the finite inputs."""
    log("relpos fp32 non-finite elements B1 S200 H2 D72")
    B, S, H, D, scale = 1, 200, 2, 72, 0.1
    qkv = seeded((B * S, 3 * H * D), 100, dtype=torch.float32)
    pd = seeded((H, 2 * S - 1), 101, std=0.02, dtype=torch.float32)
    dout = seeded((B * S, H * D), 102, dtype=torch.float32)
    out0, o32, lse = _hip.relpos_fwd(qkv, pd, B, S, H, D, scale)
    dqkv0, dpd0 = _hip.relpos_bwd(dout, qkv, pd, o32, lse, B, S, H, D, scale)
    bad = qkv.clone()
    bad[150, 2 * H * D + 5] = float("inf")  # v of key 150, head 0, dim 5
    out, _, _ = _hip.relpos_fwd(bad, pd, B, S, H, D, scale)
    assert torch.isposinf(out[:, 5]).all()  # every p is positive
    rest = torch.arange(H * D, device=out.device) != 5
    assert torch.allclose(out[:, rest], out0[:, rest], rtol=1e-5, atol=1e-6)
    assert torch.equal(out[:, D:], out0[:, D:])
    g = dout.clone()
    g[30, 7] = float("-inf")  # query 30, head 0, dim 7
    dqkv, dpd = _hip.relpos_bwd(g, qkv, pd, o32, lse, B, S, H, D, scale)
    dv, dv0 = dqkv[:, 2 * H * D:], dqkv0[:, 2 * H * D:]
    assert torch.isneginf(dv[:, 7]).all()
    rest = torch.arange(H * D, device=out.device) != 7
    assert torch.allclose(dv[:, rest], dv0[:, rest], rtol=1e-5, atol=1e-6)
    assert not torch.isfinite(dqkv[30, :D]).any()  # dq of that query: delta is infinite
    others = torch.arange(S, device=out.device) != 30
    assert torch.allclose(dqkv[others, :D], dqkv0[others, :D], rtol=1e-5, atol=1e-6)
    for i in range(3):
        assert torch.equal(dqkv[:, i * H * D + D:(i + 1) * H * D], dqkv0[:, i * H * D + D:(i + 1) * H * D])
    assert torch.equal(dpd[1], dpd0[1])


def test_relpos_fp32_very_wide_rows():
    """Row strides whose 64-row tile passes 2^31 bytes take the fp32 products (64-bit addresses)."""
    B, S, H, D, scale = 1, 3, 1, 64, 0.125
    ld = (1 << 23) + 16
    log(f"relpos fp32 row stride {ld}")
    wide = torch.zeros(S * ld, device="cuda").as_strided((S, 3 * H * D), (ld, 1))
    qkv = seeded((B * S, 3 * H * D), 110, dtype=torch.float32)
    wide.copy_(qkv)
    pd = seeded((H, 2 * S - 1), 111, dtype=torch.float32)
    dout = seeded((B * S, H * D), 112, dtype=torch.float32)
    out0, o32, lse = _hip.relpos_fwd(qkv, pd, B, S, H, D, scale)
    out, _, _ = _hip.relpos_fwd(wide, pd, B, S, H, D, scale)
    assert torch.allclose(out, out0, rtol=1e-5, atol=1e-6)
    a = _hip.relpos_bwd(dout, qkv, pd, o32, lse, B, S, H, D, scale)
    b = _hip.relpos_bwd(dout, wide, pd, o32, lse, B, S, H, D, scale)
    assert torch.allclose(a[0], b[0], rtol=1e-4, atol=1e-5) and torch.allclose(a[1], b[1], rtol=1e-4, atol=1e-5)


def test_relpos_fp32_single_products():
    """What a split leaves out of one product. At S = 1 with one nonzero column in v and dout, dpd is dp - delta,
    the split product a b minus its fp32 rounding: at most 2^-24 a b left out, and one rounding (2^-24)
    each of dp's sum and of delta. Operands whose 8 leading bits leave the largest rest, of either sign."""
    H, D = 256, 64
    log(f"relpos fp32 single products H{H} D{D}")
    i = torch.arange(H, device="cuda", dtype=torch.float64)
    u = torch.rand(2, H, generator=torch.Generator().manual_seed(140)).cuda().double()
    a = (1 + (i % 128) / 128 + (1 - u[0] / 64) * 2 ** -7).float()
    b = (1 + (7 * i % 128) / 128 + (0.5 + (u[1] - 0.5) / 64) * 2 ** -7).float()
    for x, y in ((a, a.roll(1)), (a, b), (b, b.roll(1))):
        qkv = torch.zeros(1, 3 * H * D, device="cuda")
        dout = torch.zeros(1, H * D, device="cuda")
        qkv[0, 2 * H * D + 5::D] = x
        dout[0, 5::D] = y
        pd = seeded((H, 1), 141, dtype=torch.float32)
        _, o32, lse = _hip.relpos_fwd(qkv, pd, 1, 1, H, D, 0.125)
        _, dpd = _hip.relpos_bwd(dout, qkv, pd, o32, lse, 1, 1, H, D, 0.125)
        ab = x.double() * y.double()
        assert (dpd[:, 0].double().abs() / ab).max().item() <= 3.01 * 2 ** -24


def _fp32_errors(qkv, pd, dout, B, S, H, D, scale):
    """2-norm errors of out, dq, dk, dv and dpd against float64."""
    out, o32, lse = _hip.relpos_fwd(qkv, pd, B, S, H, D, scale)
    dqkv, dpd = _hip.relpos_bwd(dout, qkv, pd, o32, lse, B, S, H, D, scale)
    r = O.relpos_manual(qkv, pd, B, S, H, D, scale, dout, compute_dtype=torch.float64)
    pairs = [(out, r[0]), *zip(dqkv.view(-1, 3, H * D).unbind(1), r[2].view(-1, 3, H * D).unbind(1)), (dpd, r[3])]
    return [((x.double() - y).norm() / y.norm()).item() for x, y in pairs]


@pytest.mark.parametrize("D", [32, 72, 128])
@pytest.mark.parametrize("v,g", [(-60, -60), (-100, 0), (0, -100), (-108, 0), (0, -118), (-118, 0), (100, 0), (0, 105)])
def test_relpos_fp32_magnitudes(D, v, g):
    """v times 2^v and dout times 2^g, down to where bf16 parts would be subnormal and up to where sums times
    2^32 overflow: a power of two commutes with every operation of fp32 products, so the errors against
    float64 stay those at 1, within a factor of two (products of splits or of fp32)."""
    B, S, H = 2, 200, 2
    log(f"relpos fp32 magnitudes D{D} v 2^{v} dout 2^{g}")
    qkv = seeded((B * S, 3 * H * D), 150, dtype=torch.float32)
    pd = seeded((H, 2 * S - 1), 151, std=0.5, dtype=torch.float32)
    dout = seeded((B * S, H * D), 152, dtype=torch.float32)
    plain = _fp32_errors(qkv, pd, dout, B, S, H, D, D ** -0.5)
    qkv[:, 2 * H * D:] *= 2.0 ** v
    errs = _fp32_errors(qkv, pd, dout * 2.0 ** g, B, S, H, D, D ** -0.5)
    assert all(e <= 2 * p for e, p in zip(errs, plain)), (errs, plain)


def test_relpos_fp32_mixed_exponents():
    """Columns of q, k and v over 15 binary orders, rows of dout over 43, and a bias that leaves keys with P
    down to 2^-126: errors against float64 within twice those of the eager fp32 computation."""
    B, S, H, D, scale = 2, 200, 2, 72, 72 ** -0.5
    log(f"relpos fp32 mixed exponents S{S} D{D}")
    gen = torch.Generator().manual_seed(160)
    qkv = seeded((B * S, 3 * H * D), 161, dtype=torch.float32)
    qkv *= 2.0 ** torch.randint(-12, 3, (3 * H * D,), generator=gen).cuda()
    dout = seeded((B * S, H * D), 162, dtype=torch.float32)
    dout *= 2.0 ** torch.randint(-40, 3, (B * S, 1), generator=gen).cuda()
    pd = -0.4 * (torch.arange(2 * S - 1, device="cuda") + 1.0).expand(H, -1).contiguous()
    errs = _fp32_errors(qkv, pd, dout, B, S, H, D, scale)
    r = O.relpos_manual(qkv, pd, B, S, H, D, scale, dout, compute_dtype=torch.float64)
    o = O.relpos_manual(qkv, pd, B, S, H, D, scale, dout)
    pairs = [(o[0], r[0]), *zip(o[2].view(-1, 3, H * D).unbind(1), r[2].view(-1, 3, H * D).unbind(1)), (o[3], r[3])]
    eager = [((x.double() - y).norm() / y.norm()).item() for x, y in pairs]
    assert all(e <= 2 * p for e, p in zip(errs, eager)), (errs, eager)


@pytest.mark.parametrize("e", [96, -96])
def test_relpos_fp32_opposite_magnitudes_of_q_and_k(e):
    """q times 2^e and k times 2^-e: the scores are those at 1, dq and dk are off by 2^-e and 2^e. Small elements
    of k or q do not split, and sums times 2^32 of the large one overflow; errors as at 1, within a factor
    of two."""
    B, S, H, D = 2, 200, 2, 72
    log(f"relpos fp32 q 2^{e} k 2^{-e}")
    qkv = seeded((B * S, 3 * H * D), 180, dtype=torch.float32)
    pd = seeded((H, 2 * S - 1), 181, std=0.5, dtype=torch.float32)
    dout = seeded((B * S, H * D), 182, dtype=torch.float32)
    plain = _fp32_errors(qkv, pd, dout, B, S, H, D, D ** -0.5)
    qkv[:, :H * D] *= 2.0 ** e
    qkv[:, H * D:2 * H * D] *= 2.0 ** -e
    errs = _fp32_errors(qkv, pd, dout, B, S, H, D, D ** -0.5)
    assert all(e <= 2 * p for e, p in zip(errs, plain)), (errs, plain)
