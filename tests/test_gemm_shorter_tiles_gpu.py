"""The ring kernel's 192x256 and 256x192 tiles (csrc/gemm_ring.h), pinned, against the 256x256 tile kernel, which sums every
element in the same order: equal bit for bit, at the tiles' edges and K tails; and the library's own choice of them."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

# (rows 1 short of, at and 1 past whole tiles; ragged columns; one K-step, two, K-steps that end inside 128 bytes)
SHAPES = [(3072, 4096, 256), (2881, 4096, 512), (3001, 4089, 544), (4096, 2880, 512), (4095, 2879, 544), (4033, 2888, 1088),
          (3001, 4096, 64), (2000, 6000, 128), (4096, 2880, 2880), (1, 1, 512), (193, 191, 800), (255, 257, 1056)]


def _operands(fmt, M, N, K, pitch_pad):
    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    if fmt != "mxfp4":
        t = [torch.randn(r, K, device="cuda", generator=g) for r in (M, N)]
        return [x.to(torch.float8_e4m3fn if fmt == "fp8" else torch.bfloat16) for x in t]
    out = []
    for r in (M, N):
        out.append(torch.randint(0, 256, (r, K // 2), dtype=torch.uint8, device="cuda", generator=g))
        out.append(torch.randint(118, 132, (r, K // 32 + pitch_pad), dtype=torch.uint8, device="cuda", generator=g))
    return out


def _gemm(lib, fmt, x, C, K, tile):
    M, N = C.shape
    s = torch.cuda.current_stream().cuda_stream
    p = [t.data_ptr() for t in x]
    if fmt == "fp8":
        return lib.hk_fp8_gemm_tile(*p, C.data_ptr(), M, N, K, 0.5, 2.0, tile, s)
    if fmt == "bf16":
        return lib.hk_bf16_gemm_tile(*p, C.data_ptr(), M, N, K, tile, s)
    return lib.hk_mxfp4_gemm_tile(p[0], p[1], x[1].shape[1], p[2], p[3], x[3].shape[1], C.data_ptr(), M, N, K, tile, s)


@pytest.mark.parametrize("fmt", ["fp8", "bf16", "mxfp4"])
@pytest.mark.parametrize("shape", SHAPES)
def test_shorter_tiles_equal_the_square_tile(hk, fmt, shape):
    M, N, K = shape
    if fmt == "mxfp4" and K < 512:
        K = 512   # (shorter scale rows that are not whole groups of 8 bytes stay with the portable kernel)
    print(f"shorter tiles {fmt} {M}x{N}x{K}", flush=True)
    lib = hk.load_library()
    for pitch_pad in ((0, 3) if fmt == "mxfp4" else (0,)):
        x = _operands(fmt, M, N, K, pitch_pad)
        buf = torch.full((3, (M * N + 575) // 64 * 64), -7.0, dtype=torch.bfloat16, device="cuda")
        for c, tile in zip(buf, (256256, 192256, 256192)):
            assert _gemm(lib, fmt, x, c[256:256 + M * N].view(M, N), K, tile) == 0
        assert torch.isfinite(buf).all()
        for c in buf[1:]:
            assert torch.equal(c.view(torch.int16), buf[0].view(torch.int16))   # the guards around C included
    assert _gemm(lib, fmt, x, buf[0][256:256 + M * N].view(M, N), K, 192192) == -6   # HK_ERR_UNSUPPORTED


@pytest.mark.parametrize("fmt", ["fp8", "bf16", "mxfp4"])
@pytest.mark.parametrize("shape,tile", [((3001, 4096, 1024), 192256), ((4096, 2880, 1024), 256192)])
def test_the_default_call_takes_them(hk, fmt, shape, tile):
    M, N, K = shape
    lib, tk = hk.load_library(), hk.tk_kernel
    assert lib.hk_gemm_tile_shape(("fp8", "bf16", "mxfp4").index(fmt), M, N, K, 1) == tile
    x = _operands(fmt, M, N, K, 0)
    C, want = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    if fmt == "fp8":
        tk.dispatch_fp8_gemm(x[0], x[1], C, 0.5, 2.0)
    elif fmt == "bf16":
        tk.dispatch_bf16_gemm(x[0], x[1], C)
    else:
        tk.dispatch_mxfp4_gemm(*x, C)
    assert _gemm(lib, fmt, x, want, K, 256256) == 0
    assert torch.isfinite(want).all() and torch.equal(C.view(torch.int16), want.view(torch.int16))
