"""The FP8-block MoE's kernel for items of up to 288 rows against the kernel for plain weights (identical bits): items of
every length, one and more per expert, every remainder of the K-steps modulo four from the shortest K on, row scales that
would show if a position took another K-step's or another row's."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _takes_tall_kernel(T, H, I, E, k):
    """The rule of moe_fp8blk_item_rows."""
    hi = T * k / E + 2 * math.sqrt(T * k / E)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rounds = lambda bm: math.ceil(E * math.ceil(hi / bm) * (I // 128) / cus)
    return min(H, I) >= 384 and 3 * rounds(288) <= 2 * min(rounds(144), rounds(160))


@pytest.mark.parametrize("T,E,k,spread", [
    (1600, 64, 8, 0.0),     # about 200 rows an expert: one item each
    (2048, 64, 8, 1.0),     # 5 to 800 rows an expert: items of every length, up to three an expert
    (1100, 64, 8, 0.3),
])
@pytest.mark.parametrize("H,I", [(384, 768), (512, 640), (640, 512), (768, 384), (896, 1152)])
def test_items_of_up_to_288_rows(hk, T, E, k, spread, H, I):
    print(f"fp8blk tall T={T} E={E} k={k} spread={spread} H={H} I={I}", flush=True)
    if not _takes_tall_kernel(T, H, I, E, k):
        pytest.skip("this device's rule takes the streaming kernel")
    assert hk.load_library().hk_moe_fp8blk_few_rows(T, H, I, E, k) == 0
    g = torch.Generator(device=DEV).manual_seed(H + T)
    e4m3 = lambda *s: (torch.randn(*s, device=DEV, generator=g) * 40).to(torch.float8_e4m3fn)
    scales = lambda *s: torch.exp2(torch.randint(-12, -4, s, device=DEV, generator=g).float())
    x, w13, w2 = e4m3(T, H), e4m3(E, 2 * I, H), e4m3(E, H, I)
    s13, s2 = scales(E, 2 * I // 128, H // 128), scales(E, H // 128, I // 128)
    xs = torch.exp2(torch.randint(-20, 8, (T, H // 128), device=DEV, generator=g).float())
    xs[5, 0], xs[17, -1], xs[T - 1, -1] = float("nan"), float("inf"), float("nan")   # neighbours must not see them
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
    clean[[5, 17, T - 1]] = False
    assert torch.isfinite(plain[clean].float()).all()
    assert torch.equal(plain[clean].view(torch.int16), shuffled[clean].view(torch.int16))
