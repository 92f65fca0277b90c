"""RMSNorm HIP kernels vs the fp32 reference on the GPU (parity tests proper)."""
import pytest
import torch

import _hip
import krsi_oracle as O
import rmsnorm as R
from krsi_testutil import assert_parity, log, seeded

pytestmark = pytest.mark.gpu
EPS = 1e-6


def _run(x, w, g, eps=EPS):
    """ref32 (fp32 autograd of the reference formula), eager bf16 original, HIP kernel."""
    ref32 = O.rmsnorm_train(x, w, eps, g.float(), torch.float32)
    orig = O.rmsnorm_train(x, w, eps, g, torch.bfloat16)
    xx = x.detach().requires_grad_(True)
    ww = w.detach().requires_grad_(True)
    y = R.rmsnorm(xx, ww, eps)
    dx, dw = torch.autograd.grad(y, [xx, ww], g)
    return ref32, orig, (y.detach(), dx, dw)


@pytest.mark.parametrize("rows", [2048, 300])
def test_rmsnorm_fwd_cpu_config(rows):
    """x [2,1024,1152] (and ragged [1,300,1152]) ~N(0,1), w ~N(1,0.02)."""
    log(f"rmsnorm fwd rows={rows} n=1152")
    x = seeded((rows, 1152), 0)
    w = seeded((1152,), 1, std=0.02, mean=1.0)
    g = seeded((rows, 1152), 2)
    ref32, orig, cand = _run(x, w, g)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand)
    # rstd against fp32, and y bitwise against eager bf16 except at rounding ties of x*r.
    import _hip

    y, rstd = _hip.rmsnorm_fwd(x, w, EPS)
    r32 = torch.rsqrt(x.float().pow(2).mean(-1) + EPS)
    assert torch.allclose(rstd, r32, rtol=2e-6, atol=0)
    same = (y == O.rmsnorm(x, w, EPS)).float().mean().item()
    assert same > 0.999, same


def test_rmsnorm_train_step_full():
    """x [8,4096,4096] fwd+bwd, y, dx and dw vs fp32 autograd."""
    log("rmsnorm fwd+bwd rows=32768 n=4096")
    x = seeded((32768, 4096), 0)
    w = seeded((4096,), 1, std=0.02, mean=1.0)
    g = seeded((32768, 4096), 2)
    ref32, orig, cand = _run(x, w, g)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand)


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 1), (5, 7), (64, 1000), (33, 1001), (17, 2048),
                                    (40, 4104), (9, 8192), (7, 12288), (5, 16384), (1000, 512)])
def test_rmsnorm_shapes(rows, n):
    log(f"rmsnorm shapes rows={rows} n={n}")
    x = seeded((rows, n), 10 + n)
    w = seeded((n,), 11, std=0.1, mean=1.0)
    g = seeded((rows, n), 12)
    ref32, orig, cand = _run(x, w, g)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand)


def test_rmsnorm_unaligned_view_takes_scalar_path():
    log("rmsnorm unaligned view")
    base = seeded((64 * 256 + 1,), 3)
    x = base[1:].view(64, 256)            # 2-byte offset: not 16-byte aligned
    w = seeded((256,), 4, std=0.1, mean=1.0)
    g = seeded((64, 256), 5)
    ref32, orig, cand = _run(x, w, g)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand)


def test_rmsnorm_empty_rows():
    x = torch.empty(0, 64, device="cuda", dtype=torch.bfloat16)
    w = seeded((64,), 1)
    xx, ww = x.requires_grad_(True), w.detach().requires_grad_(True)
    y = R.rmsnorm(xx, ww, EPS)
    assert y.shape == (0, 64)
    dx, dw = torch.autograd.grad(y, [xx, ww], torch.empty_like(y))
    assert dx.shape == (0, 64) and torch.count_nonzero(dw) == 0


def test_rmsnorm_backward_deterministic():
    log("rmsnorm determinism")
    import _hip

    x = seeded((4096, 4096), 0)
    w = seeded((4096,), 1, std=0.02, mean=1.0)
    g = seeded((4096, 4096), 2)
    _, rstd = _hip.rmsnorm_fwd(x, w, EPS)
    a = _hip.rmsnorm_bwd(g, x, w, rstd)
    b = _hip.rmsnorm_bwd(g, x, w, rstd)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_rmsnorm_deterministic_at_config2_under_interleaved_work():
    # a fixed grid of persistent workgroups writes dw partials that one
    # column-sum launch reduces in a fixed order, so runs with unrelated GPU work in between
    # (which shifts which workgroups run where and when) agree bitwise.
    import _hip

    log("rmsnorm determinism x [32768, 4096], 6 runs with interleaved work")
    x = seeded((32768, 4096), 0)
    w = seeded((4096,), 1, std=0.02, mean=1.0)
    g = seeded((32768, 4096), 2)
    first = None
    for i in range(6):
        torch.randn(1 << (16 + i), device="cuda").mul_(2).sum()
        y, rstd = _hip.rmsnorm_fwd(x, w, EPS)
        dx, dw = _hip.rmsnorm_bwd(g, x, w, rstd)
        got = (y, rstd, dx, dw)
        if first is None:
            first = [t.clone() for t in got]
        else:
            assert all(torch.equal(a, b) for a, b in zip(first, got)), f"run {i}"


def test_rmsnorm_rejects_cpu_and_wrong_dtype():
    with pytest.raises(ValueError):
        R.rmsnorm(torch.randn(4, 8, dtype=torch.bfloat16), torch.ones(8, dtype=torch.bfloat16), EPS)
    with pytest.raises(TypeError):  # float64 is not an activation dtype of the kernels
        R.rmsnorm(torch.randn(4, 8, device="cuda", dtype=torch.float64),
                  torch.ones(8, device="cuda", dtype=torch.float64), EPS)


@pytest.mark.parametrize("n", [64, 6])
def test_rmsnorm_many_short_rows(n):
    """100000 rows: the forward grid is large and the persistent backward loops ~49 times per
    row group (vector path at n = 64, scalar path at n = 6)."""
    log(f"rmsnorm rows=100000 n={n}")
    x = seeded((100000, n), 72 + n)
    w = seeded((n,), 73, std=0.1, mean=1.0)
    g = seeded((100000, n), 74)
    ref32, orig, cand = _run(x, w, g)
    assert_parity(["y", "dx", "dw"], ref32, orig, cand)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_rmsnorm_ragged_rows(dt):
    """Rows that no 16-byte chunk divides, or that start off a 16-byte boundary, from one chunk to the
    widest row of each split over the waves, against float64. Bound per element: the statistic and
    each product are fp32 sums or products of n terms, then y and dx round twice, dw once (1e-7:
    two roundings among fp16 subnormals, 2^-24 apart; the last chunk
    shares columns with the one before it, which must count once)."""
    e, u = (4 if dt == torch.float32 else 8), torch.finfo(dt).eps / 2
    for n in (e, e + 1, 2 * e - 1, 64 * e + 1, 128 * e + 3, 257 * e - 1, 512 * e + 1, 1024 * e + 5, 2048 * e - 1):
        if n > 16384:
            continue
        for off, rows in ((0, 5), (1, 3), (3, 700 if n < 300 else 2)):
            log(f"rmsnorm ragged {dt} rows={rows} n={n} offset={off}")
            x = torch.empty(rows * n + off, device="cuda", dtype=dt)[off:].view(rows, n)
            x.copy_(seeded((rows, n), 40 + n, dtype=dt))
            w, g = seeded((n,), 41, std=0.1, mean=1.0, dtype=dt), seeded((rows, n), 42, dtype=dt)
            y, rstd = _hip.rmsnorm_fwd(x, w, EPS)
            dx, dw = _hip.rmsnorm_bwd(g, x, w, rstd)
            xd, wd, gd = x.double(), w.double(), g.double()
            r = torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + EPS)
            dn = gd * wd
            ref_dx = r * dn - xd * r.pow(3) * (dn * xd).mean(-1, keepdim=True)
            s = 4e-6  # fp32 arithmetic, statistics included
            assert ((rstd.double() - r[:, 0]).abs() <= 2e-6 * r[:, 0]).all()
            assert ((y.double() - wd * xd * r).abs() <= (2.1 * u + s) * (wd * xd * r).abs() + 1e-7).all()
            mag = (r * dn).abs() + (xd * r.pow(3)).abs() * (dn * xd).abs().mean(-1, keepdim=True)
            assert ((dx.double() - ref_dx).abs() <= (2.1 * u + s) * mag + 1e-7).all()
            term = (gd * xd * r).abs().sum(0)
            assert ((dw.double() - (gd * xd * r).sum(0)).abs() <= (2.1 * u + s) * term + 1e-7).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,off", [(63, 0), (64, 1), (65, 0), (65, 3)])
def test_rmsnorm_ragged_forward_one_wave_edge(dt, n, off):
    """Ragged rows on both sides of the length that one wave holds an element per lane, where the forward
    goes over from the scalar kernel to chunks, against float64. Bounds: as above (y rounds twice)."""
    log(f"rmsnorm ragged edge {dt} n={n} offset={off}")
    u, rows = torch.finfo(dt).eps / 2, 301
    x = torch.empty(rows * n + off, device="cuda", dtype=dt)[off:].view(rows, n)
    x.copy_(seeded((rows, n), 50 + n, dtype=dt))
    w = seeded((n,), 51, std=0.1, mean=1.0, dtype=dt)
    y, rstd = _hip.rmsnorm_fwd(x, w, EPS)
    r = torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + EPS)
    ref = w.double() * x.double() * r
    assert ((rstd.double() - r[:, 0]).abs() <= 2e-6 * r[:, 0]).all()
    assert ((y.double() - ref).abs() <= (2.1 * u + 4e-6) * ref.abs() + 1e-7).all()
