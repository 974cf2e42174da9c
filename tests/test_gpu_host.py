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
