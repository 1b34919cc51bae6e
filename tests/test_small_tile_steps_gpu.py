"""The small-tile FP8 and BF16 kernels at the K-step counts where their pipeline starts, turns and ends: fewer K-steps
than LDS stages, as many, odd and even counts, with and without a partial last step; whole and ragged tiles.

Small integers: every product and sum is exact in fp32, so the result is the exact integer rounded to bf16 once."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("fmt,variant", [("fp8", 5), ("fp8", 6), ("bf16", 2), ("bf16", 3)])
@pytest.mark.parametrize("M,N", [(128, 128), (65, 200), (1, 129), (257, 64)])
def test_k_steps(hk, fmt, variant, M, N):
    per_step = 128 if fmt == "fp8" else 64
    g = torch.Generator(device=DEV).manual_seed(M + N)
    for steps in (1, 2, 3, 4, 5, 6, 7, 9, 12):
        for K in (steps * per_step, steps * per_step - per_step // 2):
            print(f"{fmt} variant {variant} M={M} N={N} K={K}", flush=True)
            a = torch.randint(-3, 4, (M, K), device=DEV, generator=g).float()
            b = torch.randint(-3, 4, (N, K), device=DEV, generator=g).float()
            dtype = torch.float8_e4m3fn if fmt == "fp8" else torch.bfloat16
            c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
            if fmt == "fp8":
                hk.tk_kernel.dispatch_fp8_gemm(a.to(dtype), b.to(dtype), c, 1.0, 1.0, variant=variant)
            else:
                hk.tk_kernel.dispatch_bf16_gemm(a.to(dtype), b.to(dtype), c, variant=variant)
            torch.cuda.synchronize()
            want = (a.cpu().double() @ b.cpu().double().T).to(torch.bfloat16)
            assert torch.equal(c.cpu(), want)
