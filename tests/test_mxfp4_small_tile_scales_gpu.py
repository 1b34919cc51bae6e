"""The scaled 64- and 128-tile kernels fetch the scales of two K-steps with the even one: every number of K-steps around the
ring of stages, odd counts, a ragged last K-step and scale rows that end inside a dword, against the portable kernel (the same
products in the same order: identical bits)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("variant", [2, 3])
@pytest.mark.parametrize("K", [512, 544, 736, 768, 1024, 1056, 1248, 1280, 1536, 1792, 2048, 2304, 2336, 2880, 4128])
def test_scales_of_every_k_step(hk, variant, K):
    M, N = 97, 200
    g = torch.Generator(device=DEV).manual_seed(K)
    # magnitudes that differ from block to block: another block's scale would show
    spread = lambda r: torch.randn(r, K, device=DEV, generator=g) * torch.exp2(
        torch.randint(-6, 7, (r, K // 32), device=DEV, generator=g).float()).repeat_interleave(32, dim=1)
    (a, sa), (b, sb) = hk.quant.quantize_mxfp4(spread(M)), hk.quant.quantize_mxfp4(spread(N))
    got, want = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    hk.tk_kernel.dispatch_mxfp4_gemm(a, sa, b, sb, got, variant=variant)
    hk.tk_kernel.dispatch_mxfp4_gemm(a, sa, b, sb, want, variant=0)
    torch.cuda.synchronize()
    assert torch.isfinite(want.float()).all()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
