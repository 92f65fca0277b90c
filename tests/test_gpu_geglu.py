"""GEGLU HIP kernels vs the fp32 reference on the GPU (parity tests proper)."""
import pytest
import torch

import _hip
import geglu as G
import krsi_oracle as O
from krsi_testutil import assert_parity, log, seeded

pytestmark = pytest.mark.gpu


def _run(u, g, approximate):
    ref32 = O.geglu_train(u, g.float(), approximate, torch.float32)
    orig = O.geglu_train(u, g, approximate, torch.bfloat16)
    uu = u.detach().requires_grad_(True)
    out = G.geglu(uu, approximate=approximate)
    (du,) = torch.autograd.grad(out, [uu], g)
    return ref32, orig, (out.detach(), du)


@pytest.mark.parametrize("approximate", ["none", "tanh"])
def test_geglu_train_step_full(approximate):
    """u [4,2048,8192] -> out [4,2048,4096], da and db vs fp32 autograd."""
    log(f"geglu fwd+bwd [8192, 8192] approximate={approximate}")
    u = seeded((8192, 8192), 0)
    g = seeded((8192, 4096), 2)
    ref32, orig, cand = _run(u, g, approximate)
    assert_parity(["out", "du"], ref32, orig, cand)
    # Forward bitwise against eager bf16, except where gelu(a) sits on a bf16 rounding tie.
    same = (cand[0] == orig[0]).float().mean().item()
    assert same > 0.999, same


@pytest.mark.parametrize("approximate", ["none", "tanh"])
@pytest.mark.parametrize("rows,f", [(1, 8), (3, 1), (7, 1001), (64, 2816), (300, 64), (2, 4100)])
def test_geglu_shapes(rows, f, approximate):
    log(f"geglu shapes rows={rows} f={f} {approximate}")
    u = seeded((rows, 2 * f), 20 + f, std=2.0)
    g = seeded((rows, f), 21)
    ref32, orig, cand = _run(u, g, approximate)
    assert_parity(["out", "du"], ref32, orig, cand)


def test_geglu_extreme_inputs_finite():
    """Large |a| saturates tanh (exp overflow path) and erf; results stay finite."""
    a = torch.tensor([-100.0, -20.0, -5.0, 0.0, 5.0, 20.0, 100.0, 3e4], device="cuda")
    u = torch.cat([a, torch.ones_like(a)]).to(torch.bfloat16)[None]
    for approx in ("tanh", "none"):
        uu = u.clone().requires_grad_(True)
        out = G.geglu(uu, approximate=approx)
        (du,) = torch.autograd.grad(out, [uu], torch.ones_like(out))
        ref = O.geglu(u.float(), approx).to(torch.bfloat16)
        assert torch.isfinite(out).all() and torch.isfinite(du).all()
        assert torch.allclose(out.float(), ref.float(), rtol=1e-2, atol=1e-2), (out, ref)


def test_geglu_deterministic():
    u = seeded((512, 4096), 0)
    g = seeded((512, 2048), 2)

    assert torch.equal(_hip.geglu_bwd(g, u), _hip.geglu_bwd(g, u))
    assert torch.equal(_hip.geglu_fwd(u), _hip.geglu_fwd(u))


def test_geglu_rejects_bad_input():
    with pytest.raises(ValueError):
        G.geglu(torch.randn(4, 8, dtype=torch.bfloat16))            # CPU tensor
    with pytest.raises(ValueError):
        G.geglu(torch.randn(4, 7, device="cuda", dtype=torch.bfloat16))  # odd width
    with pytest.raises(ValueError):
        G.geglu(torch.randn(4, 8, device="cuda", dtype=torch.bfloat16), approximate="sigmoid")


@pytest.mark.parametrize("f", [8, 3])
def test_geglu_rows_beyond_grid_y(f):
    """rows > 65535: the grid's row dimension is capped and each block strides over rows."""
    log(f"geglu rows=70000 f={f}")
    u = seeded((70000, 2 * f), 70 + f, std=2.0)
    g = seeded((70000, f), 71)
    ref32, orig, cand = _run(u, g, "tanh")
    assert_parity(["out", "du"], ref32, orig, cand)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("approximate", ["none", "tanh"])
def test_geglu_ragged_rows_match_aligned(dt, approximate):
    """Rows that no 16-byte chunk divides, or that start off a 16-byte boundary: bitwise the columns
    of the same rows padded to aligned ones (the arithmetic is per element)."""
    e = 4 if dt == torch.float32 else 8
    for f in (e, e + 1, 2 * e - 1, 257, 2048 + 1, 2730):
        log(f"geglu ragged f={f} {dt} {approximate}")
        fp = (f + e - 1) // e * e + e
        rows = 5
        up, gp = seeded((rows, 2 * fp), 30 + f, std=2.0, dtype=dt), seeded((rows, fp), 31 + f, dtype=dt)
        want, dwant = _hip.geglu_fwd(up, approximate), _hip.geglu_bwd(gp, up, approximate)
        for off in (0, 1, 3):  # elements past an aligned address
            u = torch.empty(rows * 2 * f + off, device="cuda", dtype=dt)[off:].view(rows, 2 * f)
            g = torch.empty(rows * f + off, device="cuda", dtype=dt)[off:].view(rows, f)
            u.copy_(torch.cat([up[:, :f], up[:, fp:fp + f]], dim=1))
            g.copy_(gp[:, :f])
            assert torch.equal(_hip.geglu_fwd(u, approximate), want[:, :f])
            du = _hip.geglu_bwd(g, u, approximate)
            assert torch.equal(du[:, :f], dwant[:, :f]) and torch.equal(du[:, f:], dwant[:, fp:fp + f])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("f,off", [(255, 0), (256, 1), (257, 0), (264, 3)])
def test_geglu_ragged_one_block_edge(dt, f, off):
    """Ragged rows on both sides of the width that one block covers an element per thread, where the
    kernels go over from elements to chunks: the columns of the same rows padded to aligned ones, bitwise, in
    fp16 to one ulp (the two round a product to fp32 before fp16 or at once, which differ at a tie; 2^-24: the
    subnormals' spacing)."""
    log(f"geglu ragged edge f={f} offset={off} {dt}")
    fp, rows = 272, 301
    up, gp = seeded((rows, 2 * fp), 60 + f, std=2.0, dtype=dt), seeded((rows, fp), 61 + f, dtype=dt)
    u = torch.empty(rows * 2 * f + off, device="cuda", dtype=dt)[off:].view(rows, 2 * f)
    g = torch.empty(rows * f + off, device="cuda", dtype=dt)[off:].view(rows, f)
    u.copy_(torch.cat([up[:, :f], up[:, fp:fp + f]], dim=1))
    g.copy_(gp[:, :f])
    tol = torch.finfo(dt).eps if dt == torch.float16 else 0.0
    same = lambda a, b: ((a.double() - b.double()).abs() <= tol * b.double().abs() + tol * 2.0 ** -14).all()
    for approximate in ("none", "tanh"):
        want, dwant = _hip.geglu_fwd(up, approximate), _hip.geglu_bwd(gp, up, approximate)
        assert same(_hip.geglu_fwd(u, approximate), want[:, :f])
        du = _hip.geglu_bwd(g, u, approximate)
        assert same(du[:, :f], dwant[:, :f]) and same(du[:, f:], dwant[:, fp:fp + f])
