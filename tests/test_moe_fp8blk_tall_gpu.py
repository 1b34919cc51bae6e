"""The FP8-block MoE's kernel for items of up to 288 rows against the kernel for plain weights (identical bits): items of
every length, one and more per expert, every remainder of the K-steps modulo four from the shortest K on, row scales that
would show if a position took another K-step's or another row's, numbers of choices by which a slot's number is not divided
by a shift, and the expert that every token passes through."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E,k,spread,rows", [
    (1600, 64, 8, 0.0, 288),     # about 200 rows an expert: one item each
    (2048, 64, 8, 1.0, 288),     # 5 to 800 rows an expert: items of every length, up to three an expert
    (1100, 64, 8, 0.3, 160),     # either side of the rule's line: 160 rows at mean + two standard deviations are one pass of the
    (1104, 64, 8, 0.3, 288),     # streaming kernel, 161 are two
    (1807, 64, 6, 0.3, 288),     # choices that are no power of two
    (1700, 64, 7, 1.0, 288),
])
@pytest.mark.parametrize("H,I", [(384, 768), (512, 640), (640, 512), (768, 384), (896, 1152)])
def test_items_of_up_to_288_rows(hk, T, E, k, spread, rows, H, I):
    print(f"fp8blk tall T={T} E={E} k={k} spread={spread} H={H} I={I}", flush=True)
    assert hk.load_library().hk_moe_fp8blk_item_rows(T, H, I, E, k) == rows
    g = torch.Generator(device=DEV).manual_seed(H + T)
    e4m3 = lambda *s: (torch.randn(*s, device=DEV, generator=g) * 40).to(torch.float8_e4m3fn)
    scales = lambda *s: torch.exp2(torch.randint(-12, -4, s, device=DEV, generator=g).float())
    x, w13, w2 = e4m3(T, H), e4m3(E, 2 * I, H), e4m3(E, H, I)
    s13, s2 = scales(E, 2 * I // 128, H // 128), scales(E, H // 128, I // 128)
    xs = torch.exp2(torch.randint(-20, 8, (T, H // 128), device=DEV, generator=g).float())
    # neighbours must not see them (where routing is even, the last row, whose fetch of scales ends behind the array, is a clean one)
    last = T - 1 if spread else T - 2
    xs[5, 0], xs[17, -1], xs[last, -1] = float("nan"), float("inf"), float("nan")
    logits = torch.randn(T, E, device=DEV, generator=g) + spread * torch.linspace(-2, 2, E, device=DEV)
    ws = torch.empty(hk.tk_kernel.moe_fp8blk_workspace_bytes(T, H, I, E, k), dtype=torch.uint8, device=DEV)
    ys = []
    for w in ((w13, s13, w2, s2), (hk.tk_kernel.MoeFp8BlkShuffledWeights.from_plain(w13, s13, w2, s2), None, None, None)):
        ws.fill_(0xFF)
        y = torch.zeros((T, H), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_fp8blk(x, xs, logits, None, *w, y, k, 1, 1, 2.5, ws)
        torch.cuda.synchronize()
        ys.append(y)
    plain, shuffled = ys
    clean = torch.ones(T, dtype=torch.bool, device=DEV)
    clean[[5, 17, last]] = False
    assert torch.isfinite(plain[clean].float()).all()
    assert torch.equal(plain[clean].view(torch.int16), shuffled[clean].view(torch.int16))
    # (a NaN leaves the quantization of h as a finite number; scales of zero would leave zeros)
    assert (plain[~clean] != 0).any(dim=1).all()
    assert torch.equal(plain.float().nan_to_num(nan=1e38), shuffled.float().nan_to_num(nan=1e38))


@pytest.mark.parametrize("T,H,I", [(3001, 384, 2048), (2900, 640, 2048)])   # three and five K-steps; a last item of a few rows
def test_shared_expert(hk, T, H, I):
    print(f"fp8blk tall shared T={T} H={H} I={I}", flush=True)
    assert hk.load_library().hk_moe_fp8blk_item_rows(T, H, I, 1, 1) == 288
    g = torch.Generator(device=DEV).manual_seed(T)
    e4m3 = lambda *s: (torch.randn(*s, device=DEV, generator=g) * 40).to(torch.float8_e4m3fn)
    scales = lambda *s: torch.exp2(torch.randint(-12, -4, s, device=DEV, generator=g).float())
    x, w13, w2 = e4m3(T, H), e4m3(1, 2 * I, H), e4m3(1, H, I)
    xs, s13, s2 = scales(T, H // 128), scales(1, 2 * I // 128, H // 128), scales(1, H // 128, I // 128)
    ws = torch.empty(hk.tk_kernel.moe_fp8blk_workspace_bytes(T, H, I, 1, 1), dtype=torch.uint8, device=DEV)
    ys = []
    for w in ((w13, s13, w2, s2), (hk.tk_kernel.MoeFp8BlkShuffledWeights.from_plain(w13, s13, w2, s2), None, None, None)):
        ws.fill_(0xFF)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_fp8blk_shared_expert(x, xs, *w, y, ws)
        torch.cuda.synchronize()
        ys.append(y)
    assert torch.isfinite(ys[0].float()).all()
    assert torch.equal(ys[0].view(torch.int16), ys[1].view(torch.int16))
