"""The native call path (csrc/fast.cpp) against the Python one: forms it does
not take give None (CPU), and those it takes give the general path's bits."""

import subprocess
import sys
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture
def C():
    from lockstep_amd import _capi
    return _capi


class Sub(torch.Tensor):
    pass


def test_other_forms_are_left_to_the_python_path(C):
    """CPU tensors, tensor subclasses, non-tensors and wrong argument counts."""
    x = torch.zeros(4, 128)
    u = torch.zeros(4, 64, dtype=torch.uint8)
    for bad in (x, x.as_subclass(Sub), None, 3, [1, 2]):
        assert C.fast.quantize(bad) is None and C.fast.quantize_pack(bad, True) is None
        assert C.fast.quantize_2d(bad) is None and C.fast.pack(bad) is None
        assert C.fast.quantize_pack2(bad, False) is None and C.fast.quantize_pack2([bad, bad], True) is None
        assert C.fast.linear(bad, bad, torch.float32) is None
        assert C.fast.gemm_packed(bad, u, u, u, torch.float32, False) is None
        assert C.fast.weight(bad, None, u, u, None) is None
        assert C.fast.gemm_fp8(bad, u, x, x, torch.float32, False) is None
    assert C.fast.quantize() is None and C.fast.weight(x) is None
    with pytest.raises(RuntimeError, match="gfx950 GPU only"):
        from lockstep_amd import fp4
        fp4.quantize_pack_mxfp4(x)


def test_calls_do_without_the_native_path():
    """A _fast.so that cannot be loaded (another torch, a partial build) is
    reported, and the calls run or raise as the Python path does."""
    code = """
import sys, warnings
sys.modules["lockstep_amd._fast"] = None   # import raises ImportError
with warnings.catch_warnings(record=True) as w:
    warnings.simplefilter("always")
    from lockstep_amd import fp4
assert any("_fast.so cannot be loaded" in str(x.message) for x in w)
import torch
for K, text in ((48, "multiple of block=32"), (64, "gfx950 GPU only")):
    try:
        fp4.quantize_mxfp4(torch.zeros(4, K))
    except (AssertionError, RuntimeError) as e:
        assert text in str(e), e
    else:
        raise SystemExit("no error")
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr


def test_build_makes_both_libraries(monkeypatch, tmp_path):
    """lockstep_amd.build.build() alone (the compilers replaced by a touch)."""
    from lockstep_amd import build as B
    monkeypatch.setattr(B, "PKG", tmp_path)
    monkeypatch.setattr(B, "LIB", tmp_path / "liblsmx.so")
    monkeypatch.setattr(B, "FAST_LIB", tmp_path / "_fast.so")
    monkeypatch.setattr(B, "_run", lambda cmd, verbose: Path(cmd[cmd.index("-o") + 1]).touch())
    B.build()
    assert B.LIB.exists() and B.FAST_LIB.exists()


class Recorder:
    """Passes calls to the native path and notes which of them it took."""

    def __init__(self, fast):
        self._fast, self.took = fast, []

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self._fast, name)(*a)
            self.took.append((name, r is not None))
            return r
        return call


class Declines:
    def __getattr__(self, name):
        return lambda *a: None


def _run_with(monkeypatch, C, fast, f):
    with monkeypatch.context() as m:
        m.setattr(C, "fast", fast)
        return f()


def _check(monkeypatch, C, f, native, error=None):
    """f() gives the general path's result, and its first native call takes the
    form (native), leaves it, or either (None); error: the type both raise
    instead."""
    rec = Recorder(C.fast)
    if error:
        assert not native
        for fast in (rec, Declines()):
            with pytest.raises(error):
                _run_with(monkeypatch, C, fast, f)
    else:
        assert _same(_run_with(monkeypatch, C, rec, f), _run_with(monkeypatch, C, Declines(), f))
    assert rec.took and native in (None, rec.took[0][1]), rec.took


def _same(a, b):
    if isinstance(a, (tuple, list)):
        return type(a) is type(b) and len(a) == len(b) and all(_same(x, y) for x, y in zip(a, b))
    return a.dtype == b.dtype and a.shape == b.shape and a.device == b.device and torch.equal(
        a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("R,K", [(1, 128), (3, 160), (128, 256), (257, 1152)])
def test_quantizers_match_the_python_path(C, monkeypatch, R, K, dtype):
    from lockstep_amd import fp4
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(R + K)
    base = torch.randn((R, K + 16), device=dev, generator=g).to(dtype)
    other = torch.randn((K, R + 3), device=dev, generator=g).to(dtype)
    # (rows, taken): in place with 16-byte aligned starts; other alignments,
    # other strides and empty tensors are the general path's
    for x, ok in ((base[:, :K], True), (base[:, :K].contiguous(), True), (base[:, 1:K + 1], False),
                  (other.t()[:R], False), (base[:0, :K], False)):
        # one row is contiguous wherever it starts, so no copy aligns it
        error = C.LsmxError if R == 1 and x.data_ptr() % 16 else None
        forms = [(lambda: fp4.quantize_mxfp4(x), ok), (lambda: fp4.quantize_pack_mxfp4(x), ok),
                 (lambda: fp4.quantize_pack_mxfp4_many([x, x]), ok)]
        if K % 128 == 0:
            forms.append((lambda: fp4.quantize_pack_mxfp4(x, scale_layout="kmajor"), ok))
            forms.append((lambda: fp4.quantize_pack_mxfp4_many([x, x.contiguous()], scale_layout="kmajor"), ok))
        if K % 128 == 0 and R % 128 == 0 and x.numel():
            forms.append((lambda: fp4.quantize_pack_mxfp4_2d(x), ok and dtype != torch.float32))
        for f, native in forms:
            _check(monkeypatch, C, f, native, error)
    codes = fp4.quantize_mxfp4(base[:, :K])[0]
    # an empty tensor has no storage to pass: refused
    for c, native, error in ((codes, True, None), (codes[:, :K - 32], R == 1, None), (codes[:0], False, C.LsmxError),
                             (codes.reshape(-1), False, None)):
        _check(monkeypatch, C, lambda: fp4.pack_fp4(c), native, error)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (5, 70, 384), (40, 96, 512), (130, 256, 640), (300, 1040, 2048)])
def test_products_match_the_python_path(C, monkeypatch, M, N, K):
    from lockstep_amd import dual_gemm, fp4, mxfp4_gemm
    from lockstep_amd.fp4_linear import MXFP4Linear
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, x1, w = (torch.randn(s, device=dev, generator=g) for s in ((M, K), (M, K), (N, K)))
    (xp, xk), (wp, wk) = (fp4.quantize_pack_mxfp4(t, scale_layout="kmajor") for t in (x, w))
    xr, wr = fp4.quantize_pack_mxfp4(x)[1], fp4.quantize_pack_mxfp4(w)[1]
    (xc, xs), (wc, ws) = fp4.quantize_mxfp4(x), fp4.quantize_mxfp4(w)
    odd = xs * 1.5   # scales that need the promotion
    wide = torch.zeros((M, K // 2 + 32), dtype=torch.uint8, device=dev)
    wide[:, :K // 2] = xp
    forms = []   # (call, taken by the native path, error)
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        # row-major E8M0 bytes and column-major fp32 scales are converted by the general path
        for sa, sb, ok in ((xk, wk, True), (xr, wr, False), (xs, ws, True), (xs.clone(), ws, True), (odd, ws, True),
                           (xs.t().contiguous().t(), ws, False)):
            forms.append((lambda sa=sa, sb=sb, dt=dt: mxfp4_gemm.mxfp4_gemm_packed(xp, wp, sa, sb, out_dtype=dt), ok, None))
        forms.append((lambda dt=dt: mxfp4_gemm.mxfp4_gemm_packed(wide[:, :K // 2], wp, xk, wk, out_dtype=dt), True, None))
        a, a1 = x.to(dt), x1.to(dt)
        pad = torch.zeros((M, K + 8), device=dev, dtype=dt)
        pad[:, :K] = a
        for act, rows in ((a, True), (pad[:, :K], True), (a.t().contiguous().t(), False)):
            for sw, e8m0 in ((wr, True), (ws, False)):
                ok = rows and e8m0
                forms.append((lambda act=act, sw=sw: mxfp4_gemm.mxfp4_gemm_bf16(act, wp, sw), ok, None))
                forms.append((lambda act=act, sw=sw: mxfp4_gemm.mxfp4_linear_w(act, wp, sw), ok, None))
                # both batches in one call: bf16 rows of one stride
                forms.append((lambda act=act, sw=sw, a1=a1: dual_gemm.dual_mxfp4(act, a1, wp, sw, out_dtype=torch.float32),
                              ok and dt == torch.bfloat16 and act.stride(0) == a1.stride(0), None))
        layer = MXFP4Linear(K, N).to(dev)
        layer.weight = torch.nn.Parameter(w.to(dt) if dt != torch.float16 else w)
        for t in (a, a.reshape(1, M, K)):
            forms.append((lambda layer=layer, t=t: layer(t).detach(), True, None))
    forms.append((lambda: mxfp4_gemm.mxfp4_linear_w(x1.reshape(1, M, K), wp, wr), False, None))
    forms.append((lambda: mxfp4_gemm.mxfp4_gemm_bf16(x1.double(), wp, wr), False, TypeError))
    forms.append((lambda: dual_gemm.dual_mxfp4(x.bfloat16(), x1, wp, wr), False, TypeError))
    if N % 16 == 0:
        a8, b8 = fp4.codes_to_e4m3(xc), fp4.codes_to_e4m3(wc.t().contiguous())
        wst = ws.t().contiguous()
        for sa, sb, ok in ((xs, wst, True), (odd, wst, True), (xr, wr.t().contiguous(), False)):
            forms.append((lambda sa=sa, sb=sb: mxfp4_gemm.mxfp4_gemm_fp8(a8, b8, sa, sb), ok, None))
        forms.append((lambda: mxfp4_gemm.mxfp4_gemm_fp8(a8, fp4.codes_to_e4m3(wc).t(), xs, wst), False, None))
    for f, native, error in forms:
        # one row is dense in every layout: more forms are read in place
        _check(monkeypatch, C, f, native or (None if min(M, N) == 1 else False), error)


@pytest.mark.gpu
def test_errors_are_the_python_path_s(C):
    from lockstep_amd import mxfp4_gemm
    dev = torch.device("cuda", 0)
    p = torch.zeros((4, 64), dtype=torch.uint8, device=dev)
    s = torch.full((4, 4), 127, dtype=torch.uint8, device=dev)
    with pytest.raises(AssertionError, match="multiple of 128"):
        mxfp4_gemm.mxfp4_gemm_packed(p[:, :48], p[:, :48], s, s)
    with pytest.raises(AssertionError, match="scale must be"):
        mxfp4_gemm.mxfp4_gemm_bf16(torch.zeros((2, 128), device=dev, dtype=torch.bfloat16), p, s[:, :3])
    with pytest.raises(TypeError):
        mxfp4_gemm.mxfp4_gemm_packed(p, p, s, s, out_dtype=torch.float64)
    one = torch.ones((4, 4), device=dev)
    f8 = torch.zeros((128, 128), dtype=torch.uint8, device=dev)
    for scale in (torch.full((1, 4, 4), 127, dtype=torch.uint8, device=dev), one):
        with pytest.raises(TypeError, match="unsupported dtype None"):
            mxfp4_gemm.mxfp4_gemm_packed(p, p, scale, scale, out_dtype=None)
    with pytest.raises(TypeError, match="unsupported dtype None"):
        mxfp4_gemm.mxfp4_gemm_fp8(f8[:4], f8, one, torch.ones((4, 128), device=dev), out_dtype=None)
    with pytest.raises(C.LsmxError):
        C.check(-2)


@pytest.mark.gpu
def test_calls_under_modes_and_transforms_take_the_python_path(C, monkeypatch):
    """A dispatch mode or functorch transform hands out tensors without data."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from lockstep_amd import fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    x = torch.randn((4, 128), device=dev).to(torch.bfloat16)
    pk, sc = fp4.quantize_pack_mxfp4(torch.randn((16, 128), device=dev))
    native = []

    def call():
        native.append(C.fast.quantize(x))
        native.append(C.fast.weight(x, None, pk, sc, None))
        return fp4.quantize_pack_mxfp4(x), mxfp4_gemm.mxfp4_linear_w(x, pk, sc)

    def fake():
        with FakeTensorMode(allow_non_fake_inputs=True):
            return call()

    def grad():
        return torch.func.grad(lambda s: (call()[1].float() * s).sum())(torch.ones((), device=dev))

    for f in (fake, grad):
        errors = []
        for fast in (C.fast, Declines()):
            with pytest.raises(Exception) as e:
                _run_with(monkeypatch, C, fast, f)
            errors.append((e.type, str(e.value)))
        assert errors[0] == errors[1]
    assert native and all(r is None for r in native)
    assert C.fast.quantize(x) is not None
