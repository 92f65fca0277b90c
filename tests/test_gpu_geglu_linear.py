"""The merged gate|up projection with the GEGLU epilogue fused into it (geglu_linear) against the
unfused pair the reference's geglu takes its input from (geglu.py:3-5): u = x @ w.T, then GEGLU.

Tolerance, stated: the reference's acceptance rule with slack 2 (tools/common.py:322-392,
476-518), as for every op here. Output, dx and dw are checked against the fp32 run of the unfused
pair, with the eager bf16 (or fp16) unfused pair as the yardstick, then again under
torch.compile(fullgraph=True). The fused kernel rounds the projection to the activation dtype
before the GEGLU, as the unfused pair's u tensor holds it."""
import pytest
import torch

import _hip
import geglu as G
from _harness import selftest_autograd
from krsi_testutil import log, seeded

pytestmark = pytest.mark.gpu

CASES = [  # rows, K, F, approximate, dtype
    (300, 256, 128, "tanh", torch.bfloat16),     # ragged rows: a partial row block
    (1024, 1024, 512, "none", torch.bfloat16),
    (1, 64, 64, "tanh", torch.bfloat16),
    (640, 512, 192, "tanh", torch.float16),
    (2048, 2048, 1024, "none", torch.bfloat16),
]


@pytest.mark.parametrize("rows,K,F,approximate,dt", CASES)
def test_geglu_linear_matches_unfused_pair(rows, K, F, approximate, dt):
    log(f"geglu_linear x[{rows},{K}] w[{2 * F},{K}] {approximate} {dt}")
    torch.manual_seed(0)
    x = seeded((rows, K), 0, dtype=dt)
    w = (seeded((2 * F, K), 1, dtype=torch.float32) / K ** 0.5).to(dt)
    res = selftest_autograd(lambda a, b: G.geglu_linear(a, b, approximate=approximate),
                            lambda a, b: G.reference_linear(a, b, approximate=approximate), [x, w], time=False)
    assert res["pass"], res["checks"]
    assert res["compiled"].get("pass"), res["compiled"]


def test_geglu_linear_is_the_gemm_output_rounded_then_geglu():
    """Same inputs through the fused kernel and through hipBLASLt's GEMM + the GEGLU kernel: the
    two differ only by the GEMM's summation order, so every output is within a few bf16 ulps."""
    rows, K, F = 512, 1024, 256
    x = seeded((rows, K), 3)
    w = (seeded((2 * F, K), 4, dtype=torch.float32) / K ** 0.5).to(torch.bfloat16)
    fused = G.geglu_linear(x, w)
    unfused = G.geglu(torch.nn.functional.linear(x, w))
    rel = ((fused.float() - unfused.float()).abs() / (unfused.float().abs() + 1e-2)).max().item()
    assert rel < 0.05, rel


@pytest.mark.parametrize("compiled", [False, True], ids=["eager", "compiled"])
def test_geglu_linear_frozen_weight_gets_no_gradient(compiled):
    """With the weight frozen the backward forms only dx, which equals the dx of the full
    backward bitwise (the same kernels on the same inputs)."""
    rows, K, F = 256, 512, 128
    log(f"geglu_linear frozen weight, {'compiled' if compiled else 'eager'}")
    x0 = seeded((rows, K), 5)
    w0 = (seeded((2 * F, K), 6, dtype=torch.float32) / K ** 0.5).to(torch.bfloat16)
    gy = seeded((rows, F), 7)
    fn = lambda a, b: G.geglu_linear(a, b)  # noqa: E731
    if compiled:
        torch._dynamo.reset()
        fn = torch.compile(fn, fullgraph=True)
    x, w = x0.clone().requires_grad_(True), w0.clone()
    fn(x, w).backward(gy)
    assert w.grad is None
    xf, wf = x0.clone().requires_grad_(True), w0.clone().requires_grad_(True)
    fn(xf, wf).backward(gy)
    assert torch.equal(x.grad, xf.grad) and wf.grad is not None


# Edges of the two products' tiles (128 x 128, sums in stages of 64): ragged rows, half a column tile, one, two
# and many stages, sums split over workgroups (of dx, of dw, of both, with a shorter last part) and not.
GRAD_EDGES = [  # rows, K, F
    (1, 64, 64), (63, 64, 64), (129, 192, 128), (300, 768, 2048), (64, 1024, 1408), (1000, 320, 704),
    (4099, 192, 64), (2100, 256, 576), (513, 2048, 1024),
]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,K,F", GRAD_EDGES)
def test_geglu_linear_grads_edges(rows, K, F, dt):
    """Each element within its final rounding (unit roundoff e) and the fp32 sum's bound of the float64
    result: n products of standard normal values, summed in fp32 in any order, are off by less than
    n 2^-24 times the sum of their magnitudes (about 0.64 n)."""
    log(f"geglu_linear products rows {rows} K {K} F {F} {dt}")
    du, x, w = seeded((rows, 2 * F), 1, dtype=dt), seeded((rows, K), 2, dtype=dt), seeded((2 * F, K), 3, dtype=dt)
    dx, dw = _hip.geglu_linear_grads(du, x, w)
    e = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    for got, a, b in ((dx, du, w), (dw, du.t(), x)):
        a, b = a.double(), b.double()
        ref, mag = a @ b, a.abs() @ b.abs()
        assert ((got.double() - ref).abs() <= e * ref.abs() + a.shape[1] * 2.0 ** -24 * mag + 1e-6).all()
    assert torch.equal(_hip.geglu_linear_grads(du, x, w, dw=False)[0], dx)  # the sizes alone set the order
    assert torch.equal(_hip.geglu_linear_grads(du, x, w, dx=False)[1], dw)


# Tile edges of both kernels' tiles (256 x 128 and 128 x 64): ragged rows, a last column tile half
# past F, one, two and three K stages (the staging buffers' parity carries from tile to tile), one
# and several tiles per workgroup, and one whose row count is below a tile.
EDGES = [  # rows, K, F
    (2100, 64, 2112), (2100, 128, 2112),                     # large tile, one per workgroup
    (4360, 192, 2880), (4360, 64, 2880), (4360, 256, 2880),  # large tile, two per workgroup
    (4096, 192, 2112), (4099, 128, 2112),                    # small tile, three per workgroup
    (129, 192, 64), (5, 128, 192),                           # small tile, one
]


@pytest.mark.parametrize("dt,approximate", [(torch.bfloat16, "tanh"), (torch.float16, "none")])
@pytest.mark.parametrize("rows,K,F", EDGES)
def test_geglu_linear_tile_edges(rows, K, F, dt, approximate):
    """Every output within its own rounding bound of the fp32 result: u's halves a and b, gelu(a)
    and the product each round once (unit roundoff e; |gelu'| < 1.13), and the fp32 sums of K <= 256
    products of u are off by less than 1e-4 whatever their order."""
    log(f"geglu_linear edges x[{rows},{K}] w[{2 * F},{K}] {approximate} {dt}")
    x = seeded((rows, K), 8, dtype=dt)
    w = (seeded((2 * F, K), 9, dtype=torch.float32) / K ** 0.5).to(dt)
    out = G.geglu_linear(x, w, approximate=approximate)
    a, b = (x.float() @ w.float().t()).chunk(2, dim=-1)
    ref = torch.nn.functional.gelu(a, approximate=approximate) * b
    e = torch.finfo(dt).eps / 2
    bound = 1.02 * e * (1.13 * (a * b).abs() + 3 * ref.abs()) + 1e-4 * (1.13 * b.abs() + a.abs() + 0.01)
    worst = ((out.float() - ref).abs() / bound).max().item()
    assert worst < 1, worst


@pytest.mark.parametrize("dt,approximate", [(torch.bfloat16, "none"), (torch.float16, "tanh")])
@pytest.mark.parametrize("rows,K,F", EDGES)
def test_geglu_linear_bwd_tile_edges(rows, K, F, dt, approximate):
    """du of the fused backward step, bounded as the forward above: u's halves, gelu(a), g b and the
    results round once each; |gelu'| < 1.13, |gelu''| < 0.85."""
    log(f"geglu_linear bwd edges x[{rows},{K}] w[{2 * F},{K}] {approximate} {dt}")
    x = seeded((rows, K), 10, dtype=dt)
    w = (seeded((2 * F, K), 11, dtype=torch.float32) / K ** 0.5).to(dt)
    g = seeded((rows, F), 12, dtype=dt)
    da, db = _hip.geglu_linear_bwd(g, x, w, approximate).float().chunk(2, dim=-1)
    a, b = (x.float() @ w.float().t()).chunk(2, dim=-1)
    a = a.clone().requires_grad_(True)
    gel = torch.nn.functional.gelu(a, approximate=approximate)
    (d,) = torch.autograd.grad(gel.sum(), a)
    ref_da, ref_db, e = g.float() * b * d, g.float() * gel.detach(), torch.finfo(dt).eps / 2
    g, a, b = g.float().abs(), a.detach().abs(), b.abs()
    bound_da = 1.02 * e * (0.85 * g * a * b + 3 * ref_da.abs()) + 1e-4 * g * (0.85 * b + 1.13) + 1e-6
    bound_db = 1.02 * e * (1.13 * g * a + 2 * ref_db.abs()) + 1e-4 * 1.13 * g + 1e-6
    worst = max(((da - ref_da).abs() / bound_da).max().item(), ((db - ref_db).abs() / bound_db).max().item())
    assert worst < 1, worst


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_geglu_linear_grads_of_an_empty_batch(dt):
    """rows = 0: dx is empty and dw zero, as the other entry points take an empty batch."""
    log(f"geglu_linear products of an empty batch {dt}")
    du, x, w = (torch.empty(s, device="cuda", dtype=dt) for s in ((0, 384), (0, 64), (384, 64)))
    torch.full((384, 64), 7.0, device="cuda", dtype=dt)  # what dw's memory held
    dx, dw = _hip.geglu_linear_grads(du, x, w)
    assert dx.shape == (0, 64) and dw.shape == (384, 64) and not dw.any()
