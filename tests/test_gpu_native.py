"""The native eager path of the public functions against their Python path (the autograd.Function
classes): the same kernels, so outputs and gradients are bitwise the same, over every form the
native one takes; and every form it hands back (None) still runs or raises as the Python path does."""
import pytest
import torch
from torch.autograd import forward_ad

import _hip
import geglu as G
import relpos_attention as A
import rmsnorm as R
from krsi_testutil import log, seeded

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _cases(dt):
    """(public call, Python path, native entry, inputs, whether the native path takes the call)."""
    B, S, H, D = 2, 70, 3, 72
    n = _hip.native()
    wide = seeded((B * S, 3 * H * D + 16), 4, dtype=dt)
    x, w = seeded((33, 1001), 1, dtype=dt), seeded((1001,), 2, dtype=dt)
    pd = seeded((H, 2 * S - 1), 5, dtype=torch.float32)
    bucket = A.t5_relative_position_bucket(S, True, 32, 128, pd.device)
    att = (lambda q, p: A.relpos_attention(q, p, B, S, H, D, 0.1),
           lambda q, p: A.RelPosAttention.apply(A._kernel_layout(q, H, D), p, B, S, H, D, 0.1),
           lambda q, p: n.relpos_attention(q, p, B, S, H, D, 0.1))
    cases = [
        (lambda x, w: R.rmsnorm(x, w, 1e-6), lambda x, w: R.RMSNorm.apply(x, w, 1e-6),
         lambda x, w: n.rmsnorm(x, w, 1e-6), [x, w], True),
        (lambda u: G.geglu(u, approximate="none"), lambda u: G.GEGLU.apply(u, "none"), lambda u: n.geglu(u, 0),
         [seeded((7, 2002), 3, dtype=dt)], True),
        (*att, [wide[:, :3 * H * D].contiguous(), pd], True),
        (*att, [wide, pd], True),                                # wider rows, read in place
        (*att, [wide[:, 8:8 + 3 * H * D], pd], True),            # 16-byte aligned slice
        (*att, [wide[:, 1:1 + 3 * H * D], pd], False),           # unaligned: through a copy
        (*att, [wide[:, :3 * H * D], pd.t().contiguous().t()], True),  # strided pd
        (lambda t: A.t5_relpos_table(t, S), lambda t: A.BucketTable.apply(t, bucket, S),
         lambda t: n.bucket_table(t, bucket, S), [seeded((32, H), 6, dtype=torch.float32)], True),
    ]
    if dt != torch.float32:
        xl, wl = seeded((65, 128), 7, dtype=dt), seeded((384, 128), 8, dtype=dt)
        lin = (lambda x, w: G.geglu_linear(x, w), lambda x, w: G.GEGLULinear.apply(x, w, "tanh"),
               lambda x, w: n.geglu_linear(x, w, 1))
        cases += [(*lin, [xl, wl], True), (*lin, [xl.t().contiguous().t(), wl], False)]
    return cases


def _run(fn, inputs, needs):
    leaves = [t.detach().requires_grad_(n) for t, n in zip(inputs, needs)]
    out = fn(*leaves)
    g = seeded(out.shape, 99, dtype=out.dtype)
    need = [t for t in leaves if t.requires_grad]
    return [out.detach(), *torch.autograd.grad(out, need, g)]


@pytest.mark.parametrize("dt", DTYPES)
def test_native_matches_python_path(dt):
    log(f"native against Python path {dt}")
    assert _hip.native() is not _hip._NoNative
    for fn, py, native, inputs, plain in _cases(dt):
        # The call went where the case says: a value and a C++ node, or None and the Python function's node.
        leaves = [t.detach().requires_grad_(True) for t in inputs]
        assert (native(*leaves) is not None) == plain
        assert isinstance(fn(*leaves).grad_fn, torch.autograd.function.BackwardCFunction) != plain
        assert isinstance(py(*leaves).grad_fn, torch.autograd.function.BackwardCFunction)
        patterns = [[True] * len(inputs)] + ([[True, False], [False, True]] if len(inputs) == 2 else [])
        for needs in patterns:
            for a, b in zip(_run(fn, inputs, needs), _run(py, inputs, needs)):
                assert a.stride() == b.stride() and torch.equal(a, b)
        with torch.no_grad():
            assert (native(*inputs) is not None) == plain
            a, b = fn(*inputs), py(*inputs)
        assert not a.requires_grad and torch.equal(a, b)


def test_native_saved_tensor_hooks_and_workspace_cap(monkeypatch):
    """Saved tensors pass through the default hooks, here to the CPU and back; the cap assigned
    between a forward and its backward holds for that backward."""
    log("native: saved-tensor hooks, workspace cap")
    for fn, _, _, inputs, _ in _cases(torch.bfloat16):
        needs = [True] * len(inputs)
        plain = _run(fn, inputs, needs)
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
            hooked = _run(fn, inputs, needs)
        assert packed and all(torch.equal(a, b) for a, b in zip(plain, hooked))
    B, S, H, D = 1, 700, 2, 64
    qkv, pd = seeded((B * S, 3 * H * D), 1).requires_grad_(True), seeded((H, 2 * S - 1), 2, dtype=torch.float32)
    pd.requires_grad_(True)
    out = A.relpos_attention(qkv, pd, B, S, H, D, 0.125)
    g = seeded(out.shape, 3)
    a = torch.autograd.grad(out, [qkv, pd], g, retain_graph=True)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    peaks = []
    for cap in (None, 1):
        monkeypatch.setattr(_hip, "RELPOS_BWD_WORKSPACE_MAX", cap)
        torch.cuda.reset_peak_memory_stats()
        b = torch.autograd.grad(out, [qkv, pd], g, retain_graph=True)
        peaks.append(torch.cuda.max_memory_allocated() - base)
        assert torch.equal(a[0], b[0]) and torch.allclose(a[1], b[1], rtol=1e-5, atol=1e-5)
        del b
    assert peaks[1] < peaks[0]


def test_native_backward_refuses_what_the_kernels_cannot_read(monkeypatch):
    """Saved tensors that a hook gives back elsewhere, as another type or with another shape, and a cap
    that is no number, raise in the backward, as on the Python path."""
    log("native: saved tensors given back otherwise, cap that is no number")
    hooks = [lambda t: t.cpu(), lambda t: t.double(), lambda t: t.flatten()[:-1]]
    for fn, _, _, inputs, _ in _cases(torch.bfloat16):
        for unpack in hooks:
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
                with pytest.raises((ValueError, TypeError, RuntimeError, IndexError)):
                    _run(fn, inputs, [True] * len(inputs))
    fn, py, _, inputs, _ = _cases(torch.bfloat16)[2]
    for cap in ("64", -1):
        monkeypatch.setattr(_hip, "RELPOS_BWD_WORKSPACE_MAX", cap)
        if cap == -1:  # raised to the minimum
            assert all(torch.equal(a, b) for a, b in zip(_run(fn, inputs, [True] * 2), _run(py, inputs, [True] * 2)))
        else:
            for path in (fn, py):
                with pytest.raises(TypeError):
                    _run(path, inputs, [True] * 2)


def test_native_hands_back_what_is_not_plain():
    """Tracing, functorch, duals, subclasses and refused arguments get None and so the Python path."""
    log("native: forms handed back")
    n = _hip.native()
    x, w = seeded((4, 64), 1), seeded((64,), 2)
    assert n.rmsnorm(x, w, 1e-6) is not None

    class Sub(torch.Tensor):
        pass

    class Dispatching(torch.Tensor):
        @classmethod
        def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
            raise AssertionError("not reached")

    assert n.rmsnorm(torch.nn.Parameter(x), torch.nn.Parameter(w), 1e-6) is not None
    sub = x.as_subclass(Sub)  # keeps its type, as the Python path gives it
    assert n.rmsnorm(sub, w, 1e-6) is None and type(R.rmsnorm(sub, w, 1e-6)) is type(R.RMSNorm.apply(sub, w, 1e-6))
    for args in [(x.cpu(), w.cpu(), 1e-6), (x, w.float(), 1e-6), (x[:0], w, 1e-6), (x.t(), w, 1e-6), (x, w[:32], 1e-6),
                 (x, w, 1), (x, None, 1e-6), (x, w), (x.double(), w.double(), 1e-6),
                 (torch.Tensor._make_wrapper_subclass(Dispatching, x.shape, dtype=x.dtype, device=x.device), w, 1e-6)]:
        assert n.rmsnorm(*args) is None
    with pytest.raises(TypeError):
        R.rmsnorm(x, w.float(), 1e-6)
    with pytest.raises(ValueError):
        G.geglu(seeded((4, 64), 3), approximate="gelu")
    with pytest.raises(ValueError):
        G.geglu(seeded((4, 63), 3))
    with pytest.raises(_hip.KrsiError):
        R.rmsnorm(seeded((2, 16385), 3), seeded((16385,), 4), 1e-6)
    assert R.rmsnorm(x[:0], w, 1e-6).shape == (0, 64)
    with forward_ad.dual_level():
        assert n.rmsnorm(forward_ad.make_dual(x, torch.ones_like(x)), w, 1e-6) is None
        with pytest.raises(RuntimeError):
            R.rmsnorm(forward_ad.make_dual(x, torch.ones_like(x)), w, 1e-6)
    seen = []
    for transform in (lambda f: torch.func.grad(lambda t: f(t).float().sum())(x), lambda f: torch.vmap(f)(x[None])):
        with pytest.raises(RuntimeError):
            transform(lambda t: seen.append(n.rmsnorm(t, w, 1e-6)) or R.rmsnorm(t, w, 1e-6))
    assert seen == [None, None]
    traced = []
    torch.jit.trace(lambda t: traced.append(n.rmsnorm(t, w, 1e-6)) or t * 1, (x,), check_trace=False)
    assert traced == [None]


def test_native_hands_back_nested_tensors():
    """A strided nested tensor, whose sizes and contiguity throw in C++, raises as on the Python path."""
    log("native: nested tensors")
    n = _hip.native()
    x, w = seeded((4, 128), 1), seeded((128,), 2)
    nested = torch.nested.nested_tensor([seeded((128,), 3), seeded((128,), 4)])
    f = seeded((2, 5), 5, dtype=torch.float32)
    assert n.rmsnorm(nested, w, 1e-6) is None and n.rmsnorm(x, torch.nested.nested_tensor([w]), 1e-6) is None
    assert n.geglu(nested, 1) is None and n.geglu_linear(nested, x, 1) is None
    assert n.relpos_attention(nested, f, 1, 3, 2, 8, 0.1) is None
    assert n.bucket_table(nested, x, 3) is None
    for call in (lambda: R.rmsnorm(nested, w, 1e-6), lambda: G.geglu(nested), lambda: G.geglu_linear(nested, x),
                 lambda: A.relpos_attention(nested, f, 1, 3, 2, 8, 0.1)):
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            call()


@pytest.mark.parametrize("path", ["native", "python"])
def test_native_backward_status_is_a_krsi_error(path):
    """A status that a kernel entry returns in a backward (here an output gradient off its alignment) raises
    KrsiError on both paths."""
    log(f"backward status as KrsiError: {path}")
    B, S, H, D = 1, 9, 1, 8
    qkv, pd = seeded((B * S, 3 * H * D), 1).requires_grad_(True), seeded((H, 2 * S - 1), 2, dtype=torch.float32)
    fn = A.relpos_attention if path == "native" else A.RelPosAttention.apply
    out = fn(qkv, pd, B, S, H, D, 0.1)
    g = seeded((B * S * H * D + 1,), 3)[1:].view(B * S, H * D)
    assert g.data_ptr() % 16
    with pytest.raises(_hip.KrsiError, match="aligned"):
        torch.autograd.grad(out, qkv, g)
