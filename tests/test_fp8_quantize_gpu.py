"""Per-tensor e4m3 quantization on the GPU (hk_fp8_quantize_tensor) against the torch ops of the same function on
the CPU: codes and scale are the same bits."""
import pytest
import torch

from oracle import formats as F


def _check(hk, x, ref_in=None):
    q, s = hk.quant.quantize_fp8_per_tensor(x)
    want, ws = hk.quant.quantize_fp8_per_tensor((x if ref_in is None else ref_in).cpu())
    assert isinstance(s, float) and q.shape == x.shape and q.dtype == torch.float8_e4m3fn and q.device == x.device
    assert torch.tensor(s).view(torch.int32) == torch.tensor(ws).view(torch.int32)
    assert torch.equal(q.view(torch.uint8).cpu(), want.view(torch.uint8))
    return q, s


# below, at and above: one thread's 16 elements, one block's 4096, the one-launch limit, 1024 blocks of one step
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096, 4097, 32768, 32769, 262147, 1024 * 4096, 1024 * 4096 + 5])
def test_sizes(hk, n, dtype):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, generator=g)
    x[n // 2] *= 8.0   # the maximum is one element somewhere inside
    _check(hk, x.to(dtype).cuda())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1000, 100003])
def test_special_values(hk, n):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(n, generator=g)
    _check(hk, torch.zeros(n, device="cuda"))
    for value in (float("nan"), float("-inf")):
        y = x.clone()
        y[n - 1] = value
        q, s = hk.quant.quantize_fp8_per_tensor(y.cuda())
        want, ws = hk.quant.quantize_fp8_per_tensor(y)
        assert s == ws
        # which NaN comes out of a NaN is not specified, that one does is
        got = F.e4m3_decode(q.view(torch.uint8).cpu().numpy())
        ref = F.e4m3_decode(want.view(torch.uint8).numpy())
        assert ((got == ref) | ((got != got) & (ref != ref))).all()


@pytest.mark.gpu
def test_streams_and_shapes(hk):
    xs = [torch.randn(64, 1000 + 16 * i, device="cuda").to(torch.bfloat16) for i in range(4)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    got = []
    for x, st in zip(xs, streams):
        with torch.cuda.stream(st):
            got.append(hk.quant.quantize_fp8_per_tensor(x))
    torch.cuda.synchronize()
    for x, (q, s) in zip(xs, got):
        want, ws = hk.quant.quantize_fp8_per_tensor(x.cpu())
        assert s == ws and torch.equal(q.view(torch.uint8).cpu(), want.view(torch.uint8))
    # a transposed view keeps its strides (torch ops), as before
    q, _ = _check(hk, xs[0].t())
    assert q.stride() == xs[0].t().stride()


@pytest.mark.gpu
def test_refused_under_capture(hk):
    x = torch.randn(1024, device="cuda").to(torch.bfloat16)
    hk.quant.quantize_fp8_per_tensor(x)
    torch.cuda.synchronize()
    lib = hk.load_library()
    q = torch.empty(1024, dtype=torch.uint8, device="cuda")
    ws = torch.empty(4096, dtype=torch.uint8, device="cuda")
    scale = torch.zeros(1, pin_memory=True)
    st = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        with torch.cuda.graph(graph, stream=st):
            ws.zero_()
            rc = lib.hk_fp8_quantize_tensor(x.data_ptr(), 0, 1024, q.data_ptr(), scale.data_ptr(), ws.data_ptr(), 4096,
                                            st.cuda_stream)
    assert rc == -6 and scale.item() == 0.0


def test_bad_arguments():
    from hipkittens_amd import load_library

    lib = load_library()
    a = 4096
    assert lib.hk_fp8_quantize_tensor_workspace_bytes() == 4096
    assert lib.hk_fp8_quantize_tensor(None, 0, 16, a, a, a, 4096, None) == -1
    assert lib.hk_fp8_quantize_tensor(a, 3, 16, a, a, a, 4096, None) == -2
    assert lib.hk_fp8_quantize_tensor(a, 0, 0, a, a, a, 4096, None) == -2
    assert lib.hk_fp8_quantize_tensor(a + 2, 0, 16, a, a, a, 4096, None) == -3
    assert lib.hk_fp8_quantize_tensor(a, 0, 16, a, a, a, 4095, None) == -4


class _Tagged(torch.Tensor):
    pass


def _carriers(x):
    """Functions that quantize x as something more than its memory."""
    from torch.autograd import forward_ad

    import hipkittens_amd as hk

    f = hk.quant.quantize_fp8_per_tensor
    dx = torch.linspace(-1, 1, x.numel(), device=x.device).reshape(x.shape).to(x.dtype)

    def dual():
        with forward_ad.dual_level():
            q, s = f(forward_ad.make_dual(x, dx))
            primal, tangent = forward_ad.unpack_dual(q)
            return primal.float() * s, tangent.float()

    def jvp():
        return torch.func.jvp(lambda v: f(v)[0].float(), (x,), (dx,))

    def subclass():
        q, s = f(x.as_subclass(_Tagged))
        assert type(q) is _Tagged
        return (q.as_subclass(torch.Tensor).float() * s,)

    def negated():
        q, s = f(torch._neg_view(x))
        return (q.float() * s,)

    def compiled():
        q, s = torch.compile(f, backend="eager")(x)
        return (q.float() * s,)

    return [dual, jvp, subclass, negated, compiled]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(5))
def test_tensors_that_are_more_than_their_memory(hk, i):
    x = torch.randn(48, 64, generator=torch.Generator().manual_seed(3)).cuda()
    got, want = _carriers(x)[i](), _carriers(x.cpu())[i]()
    for a, b in zip(got, want):
        assert torch.equal(a.cpu(), b)


def test_what_counts_as_plain():
    from torch.autograd import forward_ad

    from hipkittens_amd.quant import _is_plain

    x = torch.randn(4, 4)
    assert _is_plain(x) and _is_plain(x[1:]) and _is_plain(torch.nn.Parameter(x, requires_grad=False))
    assert not _is_plain(x.clone().requires_grad_()) and not _is_plain(x.as_subclass(_Tagged))
    assert not _is_plain(torch._neg_view(x))
    seen = []
    torch.func.jvp(lambda v: (seen.append(_is_plain(v)), v)[1], (x,), (x,))
    torch.func.grad(lambda v: (seen.append(_is_plain(v)), v.sum())[1])(x)
    torch.vmap(lambda v: (seen.append(_is_plain(v)), v)[1])(x)
    with forward_ad.dual_level():
        seen.append(_is_plain(forward_ad.make_dual(x, x)))
        assert _is_plain(x)
    assert seen == [False] * 4
