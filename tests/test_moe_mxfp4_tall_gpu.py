"""The MXFP4 MoE's kernel for items of up to 288 rows: every number of row fragments per item, one and more items per expert,
all epilogues, K of three K-steps and of a part of the last one. A token's result does not depend on the tokens beside it,
so the whole batch has to equal, bit for bit, the same tokens in batches small enough for the other kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows per expert: around the edges of fragments (16 and 32 rows), of the K loops (160 to 288 rows) and of items
ROWS = [0, 1, 15, 16, 17, 31, 33, 128, 159, 160, 161, 176, 177, 192, 193, 224, 225, 256, 257, 272, 273, 287, 288, 289, 305, 321,
        385, 448, 512, 576, 577, 640, 863, 865, 1000, 1152, 1153, 1700, 2000, 2500]


def _run(hk, x, logits, W, H, I, E, **options):
    T = x.shape[0]
    ws = torch.full((hk.tk_kernel.moe_mxfp4_workspace_bytes(T, H, I, E, 1),), 0xFF, dtype=torch.uint8, device=DEV)
    y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    hk.tk_kernel.dispatch_moe_mxfp4(x, logits, W, None, None, None, y, 1, ws, **options)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("biases,activation,interleaved", [
    (False, "silu", False), (True, "silu", False), (True, "swiglu_oai", True), (False, "swiglu_oai", False), (True, "silu", True)])
@pytest.mark.parametrize("H,I", [(544, 1152), (1152, 992), (768, 1056)])
def test_items_of_up_to_288_rows(hk, H, I, biases, activation, interleaved):
    print(f"mxfp4 tall H={H} I={I} {biases} {activation} {interleaved}", flush=True)
    E, T = len(ROWS), sum(ROWS)
    ext = biases or interleaved or activation != "silu"
    item_rows = lambda tokens: hk.load_library().hk_moe_mxfp4_item_rows(tokens, H, I, E, 1, 0, ext)
    assert item_rows(T) == 288 and item_rows(2048) == 192
    g = torch.Generator(device=DEV).manual_seed(H + I)
    w13 = hk.quant.quantize_mxfp4(torch.randn(E * 2 * I, H, device=DEV, generator=g) * 0.2)
    w2 = hk.quant.quantize_mxfp4(torch.randn(E * H, I, device=DEV, generator=g) * 0.2)
    pad = lambda t, rows: hk.quant.pad_scales(t.view(E, rows, -1))
    W = hk.tk_kernel.MoeMxfp4ShuffledWeights.from_plain(w13[0].view(E, 2 * I, H // 2), pad(w13[1], 2 * I),
                                                        w2[0].view(E, H, I // 2), pad(w2[1], H), interleaved=interleaved)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(ROWS, device=DEV))
    ids = ids[torch.randperm(T, device=DEV, generator=g)]
    logits = torch.zeros(T, E, device=DEV)
    logits[torch.arange(T, device=DEV), ids] = 30.0
    options = {"activation": activation}
    if biases:
        options["bias13"] = torch.randn(E, 2 * I, device=DEV, generator=g) * 2
        options["bias2"] = torch.randn(E, H, device=DEV, generator=g)
    whole = _run(hk, x, logits, W, H, I, E, **options)
    parts = [_run(hk, x[t:t + 2048], logits[t:t + 2048], W, H, I, E, **options) for t in range(0, T, 2048)]
    assert torch.isfinite(whole.float()).all()
    assert torch.equal(whole.view(torch.int16), torch.cat(parts).view(torch.int16))
