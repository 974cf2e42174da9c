"""The C++ host ops (csrc/host.cpp) against the Python ops they stand before:
the same tensors for calls that they take, None for all others, which then
meet the Python op's own checks."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


class _NoHost:
    """Host ops that take nothing: every call goes the Python way."""

    def __getattr__(self, name):
        return lambda *a: None


def _g(seed=0):
    return torch.Generator(DEV).manual_seed(seed)


def _x(*shape):
    return torch.randn(*shape, device=DEV, generator=_g(1)).half()


def _codes(*shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=_g(2))


def _scale(*shape):
    return (torch.rand(*shape, device=DEV, generator=_g(3)) * 0.01 + 1e-3).half()


def _hadk(k):
    from signrot_amd.functional import hadamard_matrices as hm
    return getattr(hm, f"get_had{k}")().half().to(DEV)


def _calls():
    """(name, thunk) of calls that the C++ ops take."""
    from signrot_amd import _CUDA as C
    from signrot_amd.functional import kernel
    K, N = 512, 96
    sign = (torch.randint(0, 2, (K,), device=DEV, generator=_g(4)) * 2 - 1).to(torch.int8)
    s28 = (torch.randint(0, 2, (14336,), device=DEV, generator=_g(5)) * 2 - 1).to(torch.int8)
    w, ws, bias = _codes(N, K // 2), _scale(N), _x(N)
    wsum = C.sum_i4(w)
    for M in (1, 5, 40, 300):
        a, sa = _codes(M, K // 2), _scale(M)
        z = torch.randint(0, 16, (M,), dtype=torch.int8, device=DEV, generator=_g(6))
        res = _x(M, N)
        yield "w4a4", lambda: C.w4a4_linear(a, sa, w, ws)
        yield "w4a4 bias", lambda: C.w4a4_linear(a, sa.view(-1, 1), w, ws.view(-1, 1), bias)
        yield "residual", lambda: C.w4a4_linear_residual(a, sa, w, ws, res, bias)
        yield "residual out", lambda: C.w4a4_linear_residual(a, sa, w, ws, res, None,
                                                             torch.zeros_like(res))
        yield "asym", lambda: C.w4a4_linear_asym(a, sa, z, w, ws, wsum, bias)
        yield "swiglu", lambda: C.w4a4_linear_swiglu(a, sa, w, ws)
        yield "quant", lambda: C.sym_quant_dynamic(_x(M, K), 0.9)
        yield "rmsnorm", lambda: C.rmsnorm_quant(_x(M, K), 1e-5, K)
        yield "head", lambda: C.head_had_quant(_x(M, 8, 128), 0.25)
        yield "had", lambda: C.had_sign_quant(_x(M, K), None, 1, sign, 1.0)
        yield "had28", lambda: C.had_sign_quant(_x(M, 14336), _hadk(28), 28, s28)
        yield "asym28", lambda: C.had_sign_asym_quant(_x(M, 14336), _hadk(28), 28, s28)
    # the split-K workspace form, and any leading dims
    big, sbig = _codes(137, 7168), _scale(137)
    wb, wbs = _codes(512, 7168), _scale(512)
    yield "split", lambda: C.w4a4_linear(big, sbig, wb, wbs)
    yield "3-D", lambda: kernel.w4a4_linear(_codes(2, 3, 256), _scale(2, 3, 1), w, ws)
    yield "3-D asym", lambda: kernel.w4a4_linear_asym(
        _codes(2, 3, 256), _scale(2, 3, 1),
        torch.ones(2, 3, 1, dtype=torch.int8, device=DEV), w, ws, wsum)
    yield "1-D", lambda: kernel.w4a4_linear(_codes(256), _scale(1), w, ws)
    yield "3-D quant", lambda: kernel.sym_quant_dynamic(_x(2, 3, K))
    yield "3-D had", lambda: kernel.had_sign_quant(_x(2, 3, K), None, 1, sign)


def _flat(r):
    return list(r) if isinstance(r, (tuple, list)) else [r]


def test_same_results(monkeypatch):
    from signrot_amd import _CUDA as C
    for name, call in _calls():
        got = _flat(call())
        with monkeypatch.context() as m:
            m.setattr(C, "_host", _NoHost())
            want = _flat(call())
        assert len(got) == len(want), name
        for a, b in zip(got, want):
            assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous(), name
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), name


def test_refused_as_before(monkeypatch):
    """Calls that the ops refuse, or take another way, do so with the C++ ops
    in front too, with the same message."""
    from signrot_amd import _CUDA as C
    from signrot_amd.functional import kernel
    a, sa, w, ws = _codes(4, 256), _scale(4), _codes(32, 256), _scale(32)
    x = _x(4, 512)
    bad = [lambda: C.w4a4_linear(a.cpu(), sa, w, ws),
           lambda: C.w4a4_linear(a.view(2, 2, 256), sa, w, ws),
           lambda: C.w4a4_linear(a, sa.float(), w, ws),
           lambda: C.w4a4_linear(a, sa[:3], w, ws),
           lambda: C.w4a4_linear(a[:, :128], sa, w, ws),
           lambda: C.w4a4_linear(a, sa, w, ws, _x(31)),
           lambda: C.w4a4_linear(None, sa, w, ws),
           lambda: C.w4a4_linear(a[:, ::2], sa, w[:, ::2], ws),
           lambda: C.w4a4_linear(_codes(4, 8), sa, _codes(32, 8), ws),     # K % 32
           lambda: C.w4a4_linear_residual(a, sa, w, ws, _x(4, 31)),
           lambda: C.w4a4_linear_swiglu(a, sa, _codes(24, 256), _scale(24)),
           lambda: C.sym_quant_dynamic(x.float()),
           lambda: C.sym_quant_dynamic(x.view(2, 2, 512)),
           lambda: C.rmsnorm_quant(_x(4, 16384), 1e-5, 16384),
           lambda: C.head_had_quant(_x(4, 12, 128), 1.0),
           lambda: C.had_sign_quant(x, None, 12),
           lambda: C.had_sign_quant(_x(2, 516), None, 1),
           lambda: C.had_sign_quant(x, None, 1, torch.ones(511, dtype=torch.int8, device=DEV)),
           lambda: kernel.w4a4_linear(a.t(), sa, w, ws)]

    def message(call):
        try:
            call()
        except Exception as e:  # noqa: BLE001
            return type(e), str(e)
        return None
    for i, call in enumerate(bad):
        got = message(call)
        with monkeypatch.context() as m:
            m.setattr(C, "_host", _NoHost())
            want = message(call)
        assert got == want and got is not None, (i, got, want)
    # taken by the Python op: no rows, a numpy clip ratio, a strided x of the module form
    import numpy as np
    assert C.sym_quant_dynamic(_x(0, 512))[0].shape == (0, 256)
    q, s = C.sym_quant_dynamic(x, np.float64(0.5))
    q2, s2 = C.sym_quant_dynamic(x, 0.5)
    assert torch.equal(q, q2) and torch.equal(s, s2)
    q, _ = kernel.sym_quant_dynamic(x.t().contiguous().t())
    assert torch.equal(q, C.sym_quant_dynamic(x)[0])


def test_current_stream():
    """Launches go to the current stream of the tensors' device."""
    from signrot_amd import _CUDA as C
    x = _x(64, 4096)
    want, _ = C.sym_quant_dynamic(x)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert C._stream(x) == side.cuda_stream
        y = torch.zeros_like(x)
        y.copy_(x)
        q, _ = C.sym_quant_dynamic(y)
        done = torch.cuda.Event()
        done.record(side)
    done.synchronize()
    assert torch.equal(q, want)


class _Recorder:
    """The real host ops, each call and whether it was taken noted."""

    def __init__(self, ops):
        self.ops, self.taken = ops, []

    def __getattr__(self, name):
        op = getattr(self.ops, name)

        def call(*a):
            out = op(*a)
            if name != "stream":
                self.taken.append(out is not None)
            return out
        return call


def test_taken_and_handed_back(monkeypatch):
    """The C++ op takes each call of _calls() at once, and none of those that
    need a second look: subclasses, functorch wrappers, fake tensors, views
    that are not contiguous, other scalars."""
    import numpy as np
    from torch._subclasses.fake_tensor import FakeTensorMode

    from signrot_amd import _CUDA as C
    from signrot_amd.functional import kernel
    rec = _Recorder(C._host)
    monkeypatch.setattr(C, "_host", rec)
    n = 0
    for name, call in _calls():
        rec.taken.clear()
        call()
        assert rec.taken == [True], name
        n += 1
    assert n == 54

    seen = []

    class Sub(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})
    x = _x(4, 512)
    a, sa, w, ws = _codes(4, 256), _scale(4), _codes(32, 256), _scale(32)
    host = rec.ops
    assert host.sym_quant_dynamic(torch.nn.Parameter(x), 1.0, 2) is not None
    handed = [lambda: host.sym_quant_dynamic(x.as_subclass(Sub), 1.0, 2),
              lambda: host.w4a4_linear(a, sa, w.as_subclass(Sub), ws, None, 2),
              lambda: host.w4a4_linear(a, sa, w, ws, _x(32).as_subclass(Sub), 2),
              lambda: host.sym_quant_dynamic(x.t(), 1.0, 2),
              lambda: host.sym_quant_dynamic(x[:, ::2], 1.0, 2),
              lambda: host.sym_quant_dynamic(x.cpu(), 1.0, 2),
              lambda: host.sym_quant_dynamic(x.float(), 1.0, 2),
              lambda: host.sym_quant_dynamic(x, np.float32(1.0), 2),
              lambda: host.sym_quant_dynamic(x, torch.ones(()), 2),
              lambda: host.sym_quant_dynamic(x, 1.0, 3),
              lambda: host.sym_quant_dynamic(x, 1.0),
              lambda: host.sym_quant_dynamic(None, 1.0, 2),
              lambda: host.sym_quant_dynamic(x[:0], 1.0, 2),
              lambda: host.sym_quant_dynamic(x.to_sparse(), 1.0, 2),
              lambda: host.had_sign_quant(x, None, 12, None, 1.0, False),
              lambda: host.had_sign_quant(x, None, 1, None, 1.0, 0),
              lambda: host.w4a4_linear(a, sa[:3], w, ws, None, 2),
              lambda: host.w4a4_linear(_codes(4, 8), sa, _codes(32, 8), ws, None, 2),
              lambda: host.w4a4_linear_residual(a, sa, w, ws, _x(4, 31), None, None)]
    for i, call in enumerate(handed):
        assert call() is None, i
    out = []
    torch.func.vmap(lambda t: out.append(host.sym_quant_dynamic(t, 1.0, 2)) or t)(_x(2, 4, 512))
    torch.func.grad(lambda t: out.append(host.sym_quant_dynamic(t, 1.0, 2)) or t.sum())(x)
    torch.func.functionalize(
        lambda t: out.append(host.sym_quant_dynamic(t, 1.0, 2)) or t)(x)
    with FakeTensorMode():
        out.append(host.sym_quant_dynamic(torch.empty(4, 512, device=DEV).half(), 1.0, 2))
    assert out == [None] * 4
    # the Python op then sees what it always saw
    seen.clear()
    q, s = kernel.sym_quant_dynamic(x.as_subclass(Sub))
    assert seen and torch.equal(q, host.sym_quant_dynamic(x, 1.0, 2)[0])


_STUB = """
int stub_rc = 0, stub_calls = 0;
%s
long long srq_w4a4_linear_ws_bytes() { return 0; }
int srq_w4a4_linear_asym_ws_bytes(long long M, long long N, long long K, long long *b)
{ return *b = 0; }
const char *srq_last_error() { return "stub"; }
"""

_CHILD = """
import ctypes, importlib.machinery, importlib.util, pathlib, sys
import torch
from signrot_amd import _native
from signrot_amd._native import NativeError
here = pathlib.Path(sys.argv[1])
stub = ctypes.CDLL(str(here / "libsignrot_hip.so"), mode=ctypes.RTLD_GLOBAL)
rc, calls = (ctypes.c_int.in_dll(stub, n) for n in ("stub_rc", "stub_calls"))
loader = importlib.machinery.ExtensionFileLoader("srq_host", str(here / "srq_host.so"))
host = importlib.util.module_from_spec(importlib.util.spec_from_loader("srq_host", loader))
loader.exec_module(host)
u8 = lambda *s: torch.zeros(s, dtype=torch.uint8, device="cuda")
f16 = lambda *s: torch.zeros(s, dtype=torch.float16, device="cuda")
i8 = torch.zeros(2, dtype=torch.int8, device="cuda")
i32 = torch.zeros(32, dtype=torch.int32, device="cuda")
res = f16(2, 32)
ops = [(host.had_sign_quant, (f16(2, 64), None, 1, None, 1.0, False)),
       (host.had_sign_asym_quant, (f16(2, 64), None, 1, None, 1.0, True)),
       (host.had_sign_asym_quant, (f16(2, 64), None, 1, None, 1.0, False)),
       (host.sym_quant_dynamic, (f16(2, 64), 1.0, 2)),
       (host.rmsnorm_quant, (f16(2, 64), 1e-5, 64, 1.0)),
       (host.head_had_quant, (f16(2, 8, 16), 1.0, 1.0)),
       (host.w4a4_linear, (u8(2, 32), f16(2), u8(32, 32), f16(32), None, 2)),
       (host.w4a4_linear_residual, (u8(2, 32), f16(2), u8(32, 32), f16(32), res, None, res)),
       (host.w4a4_linear_asym, (u8(2, 32), f16(2), i8, u8(32, 32), f16(32), i32, None, 2)),
       (host.w4a4_linear_swiglu, (u8(2, 32), f16(2), u8(32, 32), f16(32)))]
for op, args in ops:
    name = op.__name__
    for code, outcome in ((0, "result"), (-1, None), (-2, None), (-3, "raises"), (-9, "raises")):
        rc.value, before = code, calls.value
        try:
            got = op(*args)
            got = None if got is None else "result"
        except NativeError as e:
            got = "raises"
            assert f"({code}): stub" in str(e) and name in str(e), (name, str(e))
        assert got == outcome, (name, code, got)
        assert calls.value == before + 1, (name, code)
print("ok", flush=True)
"""


def test_failed_launch_is_raised_once(tmp_path):
    """A launch error of the library is raised and the call not repeated by
    the Python op (an in-place residual would be added twice); an argument
    that the library refuses goes to the Python op.  The real extension over a
    stub of the library that only counts calls: nothing runs on the GPU."""
    import pathlib
    import shutil
    import subprocess
    import sys

    import signrot_amd
    from signrot_amd import _native
    root = pathlib.Path(signrot_amd.__file__).resolve().parents[1]
    entries = [n for n in _native.SIGNATURES if not n.endswith("_ws_bytes")]
    (tmp_path / "stub.c").write_text(_STUB % "\n".join(
        f"int {n}() {{ ++stub_calls; return stub_rc; }}" for n in entries))
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(tmp_path / "libsignrot_hip.so"),
                    str(tmp_path / "stub.c")], check=True)
    shutil.copy(_native.HOST_PATH, tmp_path / "srq_host.so")
    (tmp_path / "child.py").write_text(_CHILD)
    run = subprocess.run([sys.executable, str(tmp_path / "child.py"), str(tmp_path)], cwd=root,
                         env={**__import__("os").environ, "PYTHONPATH": str(root)},
                         capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), run.stderr[-2000:]
