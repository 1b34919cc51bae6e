"""The ring kernel's 192x256 and 256x192 tiles (csrc/gemm_ring.h, chosen by pick_shorter_tile) against the 256x256
tile kernel, which sums every element in the same order: equal bit for bit, at the tiles' edges and K tails."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

# (rows 1 short of, at and 1 past whole tiles; ragged columns; one K-step, two, K-steps that end inside 128 bytes)
SHAPES = [(3072, 4096, 256), (2881, 4096, 512), (3001, 4089, 544), (4096, 2880, 512), (4095, 2879, 544), (4033, 2888, 1088),
          (3001, 4096, 64), (2000, 6000, 128), (4096, 2880, 2880)]


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


@pytest.mark.parametrize("fmt", ["fp8", "bf16", "mxfp4"])
@pytest.mark.parametrize("shape", SHAPES)
def test_shorter_tiles_equal_the_square_tile(fmt, shape):
    from hipkittens_amd import _lib, tk_kernel as tk

    M, N, K = shape
    if fmt == "mxfp4" and K < 512:
        K = 512   # (shorter scale rows that are not whole groups of 8 bytes stay with the portable kernel)
    code = {"fp8": 0, "bf16": 1, "mxfp4": 2}[fmt]
    picked = _lib.load_library().hk_gemm_shorter_tile(code, M, N, K)
    print(f"shorter tiles {fmt} {M}x{N}x{K}: {picked}", flush=True)
    assert picked == (2 if M > 4000 or N == 6000 else 1)
    for pitch_pad in ((0, 3) if fmt == "mxfp4" else (0,)):
        x = _operands(fmt, M, N, K, pitch_pad)
        buf = torch.full((2, (M * N + 575) // 64 * 64), -7.0, dtype=torch.bfloat16, device="cuda")
        for c, variant in ((buf[0], -1), (buf[1], {"fp8": 4}.get(fmt, 1))):
            C = c[256:256 + M * N].view(M, N)
            if fmt == "fp8":
                tk.dispatch_fp8_gemm(x[0], x[1], C, 0.5, 2.0, variant=variant)
            elif fmt == "bf16":
                tk.dispatch_bf16_gemm(x[0], x[1], C, variant=variant)
            elif pitch_pad and variant == 1:   # the pinned form takes dense scale rows
                nb = K // 32
                tk.dispatch_mxfp4_gemm(x[0], x[1][:, :nb].contiguous(), x[2], x[3][:, :nb].contiguous(), C, variant=1)
            else:
                tk.dispatch_mxfp4_gemm(*x, C, variant=variant)
        assert torch.isfinite(buf).all()
        assert torch.equal(buf[0].view(torch.int16), buf[1].view(torch.int16))   # the guards around C included
