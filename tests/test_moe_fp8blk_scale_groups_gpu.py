"""The FP8-block streaming kernel fetches an activation row's scales four K-steps at a time: every remainder of the
K-steps modulo four and rows shorter than one group, against the kernel for plain weights (identical bits), with scales that
would show if a position took another K-step's or another row's."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E", [(1000, 4), (1500, 12)])   # several items an expert, and about two (items of 144 or 160 rows)
@pytest.mark.parametrize("H", [128, 256, 384, 512, 640, 768, 896, 1024, 1152])
def test_row_scales_in_groups_of_four(hk, T, E, H):
    I, k = 512, 2
    print(f"fp8blk scale groups T={T} E={E} H={H}", flush=True)
    assert hk.load_library().hk_moe_fp8blk_item_rows(T, H, I, E, k) in (144, 160)   # the streaming kernel
    g = torch.Generator(device=DEV).manual_seed(H + E)
    e4m3 = lambda *s: (torch.randn(*s, device=DEV, generator=g) * 40).to(torch.float8_e4m3fn)
    scales = lambda *s: torch.exp2(torch.randint(-12, -4, s, device=DEV, generator=g).float())
    x, w13, w2 = e4m3(T, H), e4m3(E, 2 * I, H), e4m3(E, H, I)
    s13, s2 = scales(E, 2 * I // 128, H // 128), scales(E, H // 128, I // 128)
    xs = torch.exp2(torch.randint(-20, 8, (T, H // 128), device=DEV, generator=g).float())
    xs[5, 0], xs[17, -1], xs[T - 1, -1] = float("nan"), float("inf"), float("nan")   # neighbours must not see them
    logits = torch.randn(T, E, device=DEV, generator=g)
    ws = torch.empty(hk.tk_kernel.moe_fp8blk_workspace_bytes(T, H, I, E, k), dtype=torch.uint8, device=DEV)
    ys = []
    for w in ((w13, s13, w2, s2), (hk.tk_kernel.MoeFp8BlkShuffledWeights.from_plain(w13, s13, w2, s2), None, None, None)):
        y = torch.zeros((T, H), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_fp8blk(x, xs, logits, None, *w, y, k, 1, 1, 2.5, ws)
        torch.cuda.synchronize()
        ys.append(y)
    plain, shuffled = ys
    clean = torch.ones(T, dtype=torch.bool, device=DEV)
    clean[[5, 17, T - 1]] = False
    assert torch.isfinite(plain[clean].float()).all()
    assert torch.equal(plain[clean].view(torch.int16), shuffled[clean].view(torch.int16))
    assert torch.equal(plain.isnan(), shuffled.isnan())
