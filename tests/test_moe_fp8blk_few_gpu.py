"""The few-rows kernel of the FP8 block-scaled MoE (decode steps, shared expert; pre-shuffled weights) against the plain
weight layout's LDS-staged kernel: same MFMAs, K order and scaling FMAs, so the outputs agree bit for bit. (The plain
layout is compared with the oracle in test_moe_fp8blk_gpu.py.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(hk, T, E, H, I, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g)
    w13 = torch.empty((E, 2 * I, H), dtype=torch.float8_e4m3fn, device=DEV)
    s13 = torch.empty((E, 2 * I // 128, H // 128), device=DEV)
    w2 = torch.empty((E, H, I), dtype=torch.float8_e4m3fn, device=DEV)
    s2 = torch.empty((E, H // 128, I // 128), device=DEV)
    for e in range(E):
        w13[e], s13[e] = hk.quant.quantize_fp8_blocks(rn(2 * I, H) * 0.1, 128, 128)
        w2[e], s2[e] = hk.quant.quantize_fp8_blocks(rn(H, I) * 0.1, 128, 128)
    xq, xs = hk.quant.quantize_fp8_blocks(rn(T, H), 1, 128)
    return xq, xs, rn(T, E), (w13, s13, w2, s2)


# K-steps of gate+up = H / 128, of down = I / 128: fewer than, as many as and more than the ring's seven; an odd
# number of 128-column blocks of H; experts with 15 to 17 rows and more; the rule's edges on 256 CUs, each followed by a
# layer beyond it that takes the streaming kernel (2 rows per expert; 3/4 of an item per CU; 192 rows per expert)
STREAMING = {(129, 64, 1, 256, 2048), (320, 2, 1, 256, 1152), (385, 2, 1, 256, 896)}


@pytest.mark.parametrize("T,E,k,H,I", [(1, 8, 8, 128, 128), (3, 16, 4, 768, 896), (16, 64, 8, 896, 1024),
                                       (33, 16, 1, 1024, 128), (15, 2, 1, 1152, 256), (32, 2, 1, 256, 384),
                                       (34, 2, 2, 384, 640), (380, 2, 1, 256, 896), (384, 2, 1, 256, 896),
                                       (385, 2, 1, 256, 896), (319, 2, 1, 256, 1152), (320, 2, 1, 256, 1152),
                                       (128, 64, 1, 256, 2048), (129, 64, 1, 256, 2048),
                                       (20, 16, 4, 640, 512), (20, 16, 4, 512, 640)])   # rings of four and seven K-steps
def test_routed_layer_has_the_bits_of_the_plain_layout(hk, T, E, k, H, I):
    print(f"fp8blk few T={T} E={E} k={k} H={H} I={I}", flush=True)
    tk = hk.tk_kernel
    assert hk.load_library().hk_moe_fp8blk_few_rows(T, H, I, E, k) == (0 if (T, E, k, H, I) in STREAMING else 16)
    xq, xs, logits, plain = _layer(hk, T, E, H, I, T + E + H)
    ws = torch.empty(tk.moe_fp8blk_workspace_bytes(T, H, I, E, k), dtype=torch.uint8, device=DEV)
    out = []
    for weights in (plain, (tk.MoeFp8BlkShuffledWeights.from_plain(*plain), None, None, None)):
        ws.fill_(0xFF)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        tk.dispatch_moe_fp8blk(xq, xs, logits, None, *weights, y, k, 1, 1, 1.0, ws)
        out.append(y)
    torch.cuda.synchronize()
    assert torch.isfinite(out[0].float()).all()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("T,H,I", [(1, 128, 128), (15, 896, 256), (16, 1024, 896), (17, 384, 1024), (191, 256, 1920),
                                   (192, 256, 1920), (193, 256, 1920), (400, 512, 384)])
def test_shared_expert_has_the_bits_of_the_plain_layout_and_of_the_routed_call(hk, T, H, I):
    print(f"fp8blk shared T={T} H={H} I={I}", flush=True)
    tk = hk.tk_kernel
    # few rows up to 3/4 of an item per CU (I = 1920: 191 tokens) and 192 rows
    assert hk.load_library().hk_moe_fp8blk_few_rows(T, H, I, 1, 1) == (16 if T < 192 else 0)
    xq, xs, _, plain = _layer(hk, T, 1, H, I, T + H)
    ws = torch.empty(tk.moe_fp8blk_workspace_bytes(T, H, I, 1, 1), dtype=torch.uint8, device=DEV)
    shuffled = (tk.MoeFp8BlkShuffledWeights.from_plain(*plain), None, None, None)
    ident = torch.arange(T, dtype=torch.int32, device=DEV)
    want = torch.empty((T, H), dtype=torch.bfloat16, device=DEV)
    tk.dispatch_moe_fp8blk_experts(xq, xs, *plain, torch.ones((T, 1), device=DEV), ident,
                                   torch.tensor([0, T], dtype=torch.int32, device=DEV), ident, want, ws)
    for weights in (plain, shuffled):
        ws.fill_(0xFF)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        tk.dispatch_moe_fp8blk_shared_expert(xq, xs, *weights, y, ws)
        assert torch.equal(y, want)
    assert torch.isfinite(want.float()).all()
    two = [w.repeat(2, 1, 1) for w in plain]
    with pytest.raises(RuntimeError):   # one expert's weights
        tk.dispatch_moe_fp8blk_shared_expert(xq, xs, *two, y, ws)
