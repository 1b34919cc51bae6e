"""The native dispatchers (csrc/dispatch.cpp): they take what the Python dispatchers take, leave the rest to them, and give
the same results."""
import warnings
from pathlib import Path

import pytest
import torch

import hipkittens_amd as hk
from hipkittens_amd import _lib

tk = hk.tk_kernel


def _needs_build():
    if not hk.lib_path().exists():
        pytest.skip("library not built")


def test_cpu_tensors_and_wrong_types_are_left_to_python():
    _needs_build()
    nat = _lib.load_dispatch()
    a, c = torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(4, 4, dtype=torch.bfloat16)
    u = torch.zeros(4, 64, dtype=torch.uint8)
    assert nat.bf16_gemm(a, a, c, None) is None
    assert nat.fp8_gemm(u, u, c, 1.0, 1.0, None) is None
    assert nat.mxfp4_gemm(u, u, u, u, c, None) is None
    assert nat.mxfp4_quantize_rows(a, u, u) is None
    assert nat.bf16_gemm(a, a, c) is None and nat.bf16_gemm(None, 3, "x", a) is None
    with pytest.raises(RuntimeError, match="GPU device"):
        tk.dispatch_bf16_gemm(a, a, c)
    with pytest.raises(RuntimeError, match="expected a torch.Tensor"):
        tk.dispatch_fp8_gemm([1], u, c)


def _python_only(monkeypatch, path="/nonexistent/_dispatch.so"):
    monkeypatch.setattr(_lib, "_DISPATCH_PATH", Path(path))
    monkeypatch.setattr(_lib, "_dispatch", None)
    monkeypatch.setattr(tk, "_native", None)


@pytest.mark.parametrize("how", ["absent", "not a module", "another torch"])
def test_without_the_module_the_python_dispatchers_take_every_call(monkeypatch, tmp_path, how):
    """What the module does not load for (it is missing, broken, or compiled against another torch) is no call's failure."""
    _needs_build()
    built = _lib._DISPATCH_PATH
    (tmp_path / "_dispatch.so").write_text("no shared object")
    _python_only(monkeypatch, {"absent": tmp_path / "none.so", "not a module": tmp_path / "_dispatch.so"}.get(how, built))
    if how == "another torch":
        monkeypatch.setattr(torch, "__version__", "0.1")
    with pytest.raises((RuntimeError, ImportError)):
        _lib.load_dispatch()
    a, c = torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(4, 4, dtype=torch.bfloat16)
    u = torch.zeros(4, 64, dtype=torch.uint8)
    calls = [lambda: tk.dispatch_bf16_gemm(a, a, c), lambda: tk.dispatch_fp8_gemm(u, u, c),
             lambda: tk.dispatch_mxfp4_gemm(u, u, u, u, c), lambda: tk.dispatch_mxfp4_quantize_rows(a, u, u)]
    for i, call in enumerate(calls):
        with warnings.catch_warnings(record=True) as said:
            warnings.simplefilter("always")
            with pytest.raises(RuntimeError, match="GPU device"):   # the Python dispatcher's own check
                call()
        assert [w.category for w in said] == ([RuntimeWarning] if i == 0 else [])   # said once


def test_the_build_goes_on_without_a_host_compiler(monkeypatch, tmp_path, capsys):
    from hipkittens_amd import build

    def no_compiler():
        raise FileNotFoundError("g++")

    stale = tmp_path / "_dispatch.so"
    stale.write_text("of an earlier build")
    monkeypatch.setattr(build, "DISPATCH_PATH", stale)
    monkeypatch.setattr(build, "_build_dispatch", no_compiler)
    monkeypatch.setattr(build, "_compile_one", lambda src, extra: src)
    linked = []
    monkeypatch.setattr(build, "_link", lambda objs, out: linked.append(out))
    assert build.build(check=False) == build.LIB_PATH and build.LIB_PATH in linked
    assert not stale.exists() and "not built" in capsys.readouterr().err


def _calls(dev):
    g = torch.Generator(device=dev).manual_seed(3)
    M, N, K = 33, 80, 544
    x, w = (torch.randn(r, K, device=dev, generator=g).to(torch.bfloat16) for r in (M, N))
    (x8, sx), (w8, sw) = hk.quant.quantize_fp8_per_tensor(x), hk.quant.quantize_fp8_per_tensor(w)
    (x4, xs), (w4, ws) = hk.quant.quantize_mxfp4(x), hk.quant.quantize_mxfp4(w)
    pad, space = hk.quant.pad_scales(xs), torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    new = lambda: torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    q = lambda: (torch.zeros(M, K // 2, dtype=torch.uint8, device=dev), torch.zeros(M, 24, dtype=torch.uint8, device=dev))
    return {
        "fp8": (tk.dispatch_fp8_gemm, lambda c: (x8, w8, c, sx, sw), {}, new),
        "fp8 bytes": (tk.dispatch_fp8_gemm, lambda c: (x8.view(torch.uint8), w8, c), {}, new),
        "fp8 int scales": (tk.dispatch_fp8_gemm, lambda c: (x8, w8, c, 2, 1), {}, new),   # (left to Python)
        "fp8 workspace": (tk.dispatch_fp8_gemm, lambda c: (x8, w8, c, sx, sw), {"workspace": space}, new),
        "bf16": (tk.dispatch_bf16_gemm, lambda c: (x, torch.nn.Parameter(w), c), {}, new),
        "bf16 workspace": (tk.dispatch_bf16_gemm, lambda c: (x, w, c), {"workspace": space}, new),
        "mxfp4": (tk.dispatch_mxfp4_gemm, lambda c: (x4, xs, w4, ws, c), {}, new),
        "mxfp4 e8m0": (tk.dispatch_mxfp4_gemm, lambda c: (x4, xs.view(torch.float8_e8m0fnu), w4, ws, c), {}, new),
        "mxfp4 pitched": (tk.dispatch_mxfp4_gemm, lambda c: (x4, pad, w4, ws, c), {}, new),
        "mxfp4 workspace": (tk.dispatch_mxfp4_gemm, lambda c: (x4, pad, w4, ws, c), {"workspace": space}, new),
        "quantize": (tk.dispatch_mxfp4_quantize_rows, lambda o: (x, *o), {}, q),
    }


_NAMES = ["fp8", "fp8 bytes", "fp8 int scales", "fp8 workspace", "bf16", "bf16 workspace", "mxfp4", "mxfp4 e8m0",
          "mxfp4 pitched", "mxfp4 workspace", "quantize"]


def _same(a, b):
    flat = lambda o: [t.view(torch.uint8) for t in (o if isinstance(o, tuple) else (o,))]
    return all(torch.equal(x, y) for x, y in zip(flat(a), flat(b)))


@pytest.mark.gpu
@pytest.mark.parametrize("name", _NAMES)
def test_same_results_as_the_python_dispatcher(monkeypatch, name):
    fn, args, kw, new = _calls("cuda:0")[name]
    out = [new(), new()]
    fn(*args(out[0]), **kw)
    torch.cuda.synchronize()
    _python_only(monkeypatch)
    with pytest.warns(RuntimeWarning, match="in Python"):
        fn(*args(out[1]), **kw)
    torch.cuda.synchronize()
    assert _same(out[0], out[1])
    assert not isinstance(out[0], torch.Tensor) or torch.isfinite(out[0].float()).all()


@pytest.mark.gpu
def test_refused_as_before():
    dev = "cuda:0"
    a = torch.zeros(32, 64, dtype=torch.bfloat16, device=dev)
    c = torch.zeros(32, 32, dtype=torch.bfloat16, device=dev)
    u = torch.zeros(32, 64, dtype=torch.uint8, device=dev)
    for bad in [lambda: tk.dispatch_bf16_gemm(a, a, c[:, :16]), lambda: tk.dispatch_bf16_gemm(a.t(), a, c),
                lambda: tk.dispatch_bf16_gemm(a, a.cpu(), c), lambda: tk.dispatch_bf16_gemm(a, a.float(), c),
                lambda: tk.dispatch_bf16_gemm(a.view(-1)[4:4 + 32 * 60].view(32, 60), a[:, :60].contiguous(), c),
                lambda: tk.dispatch_fp8_gemm(u, u[:, :48].contiguous(), c), lambda: tk.dispatch_fp8_gemm(u, u, c, workspace=a),
                lambda: tk.dispatch_mxfp4_gemm(u, u[:, :2], u, u, c), lambda: tk.dispatch_mxfp4_gemm(u, u[:16], u, u, c),
                lambda: tk.dispatch_mxfp4_quantize_rows(a, u, u),
                lambda: torch.vmap(lambda t: tk.dispatch_bf16_gemm(t, a, c))(a.unsqueeze(0))]:
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.gpu
@pytest.mark.parametrize("name", _NAMES)
def test_the_current_stream_is_used(name):
    """The call waits for what its own stream does to an operand: milliseconds of products, then the operand's final
    values. On another stream it would see the values from before."""
    fn, args, kw, new = _calls("cuda:0")[name]
    outs = [new() for _ in range(3)]   # of the first values, of the final ones, from the side stream
    a = args(outs[0])[0].view(torch.uint8)
    first, final = a.clone(), a.flip(0).contiguous()
    for values, out in zip((first, final), outs):
        a.copy_(values)
        fn(*args(out), **kw)
    a.copy_(first)
    busy = torch.randn(4096, 4096, device="cuda:0")
    torch.cuda.synchronize()
    assert not _same(outs[0], outs[1])
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(8):
            torch.mm(busy, busy)
        a.copy_(final)
        fn(*args(outs[2]), **kw)
    side.synchronize()
    assert _same(outs[2], outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("name", _NAMES)
def test_captured_calls_replay(name):
    fn, args, kw, new = _calls("cuda:0")[name]
    want, got = new(), new()
    fn(*args(want), **kw)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn(*args(got), **kw)
    for _ in range(3):
        for t in got if isinstance(got, tuple) else (got,):
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert _same(got, want)
