"""The streaming MXFP4 MoE kernel where several work items share an expert: every number of row fragments per item, both
activations, MXFP4 and MXFP8 rows. A token's result does not depend on the tokens beside it, so the whole batch has to
equal, bit for bit, the same tokens in batches small enough for the other kernels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows per expert: around the edges of fragments (16 rows), of the fragments under one branch (80, 96 and 128 rows for items of
# up to 128, 144 and 192) and of items (128, 144, 192); the mean has to stay above one item
ROWS = [1, 16, 17, 63, 65, 79, 80, 81, 95, 96, 97, 112, 113, 127, 128, 129, 144, 145, 176, 177, 191, 192, 193, 208, 288, 384,
        385, 400, 577, 900]


def _layer(hk, E, H, I, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w13 = hk.quant.quantize_mxfp4(torch.randn(E * 2 * I, H, device=DEV, generator=g) * 0.2)
    w2 = hk.quant.quantize_mxfp4(torch.randn(E * H, I, device=DEV, generator=g) * 0.2)
    pad = lambda t, rows: hk.quant.pad_scales(t.view(E, rows, -1))
    W = hk.tk_kernel.MoeMxfp4ShuffledWeights.from_plain(w13[0].view(E, 2 * I, H // 2), pad(w13[1], 2 * I),
                                                        w2[0].view(E, H, I // 2), pad(w2[1], H))
    return g, W


def _run(hk, x, logits, W, H, I, E, act_format, **options):
    T = x.shape[0]
    ws = torch.empty(hk.tk_kernel.moe_mxfp4_workspace_bytes(T, H, I, E, 1, act_format), dtype=torch.uint8, device=DEV)
    y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    hk.tk_kernel.dispatch_moe_mxfp4(x, logits, W, None, None, None, y, 1, ws, act_format=act_format, **options)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("act_format", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("biases,activation", [(False, "silu"), (True, "silu"), (True, "swiglu_oai"), (False, "swiglu_oai")])
@pytest.mark.parametrize("H,I", [(512, 288), (1056, 128)])
def test_rows_of_every_fragment_count(hk, H, I, biases, activation, act_format):
    print(f"moe row groups H={H} I={I} {biases} {activation} {act_format}", flush=True)
    E, T = len(ROWS), sum(ROWS)
    g, W = _layer(hk, E, H, I, H + I)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(ROWS, device=DEV))
    ids = ids[torch.randperm(T, device=DEV, generator=g)]
    logits = torch.zeros(T, E, device=DEV)
    logits[torch.arange(T, device=DEV), ids] = 30.0
    options = {"activation": activation}
    if biases:
        options["bias13"] = torch.randn(E, 2 * I, device=DEV, generator=g) * 2
        options["bias2"] = torch.randn(E, H, device=DEV, generator=g)
    whole = _run(hk, x, logits, W, H, I, E, act_format, **options)
    parts = [_run(hk, x[t:t + 640], logits[t:t + 640], W, H, I, E, act_format, **options) for t in range(0, T, 640)]
    assert torch.isfinite(whole.float()).all()
    assert torch.equal(whole.view(torch.int16), torch.cat(parts).view(torch.int16))


@pytest.mark.parametrize("T", [64, 1024])   # one item an expert, and several
def test_clamped_swiglu_of_nan(hk, T):
    """A NaN reaches the clamps as fmin / fmax treat it: gate -> limit, up -> -limit."""
    H, I, E = 256, 128, 2
    g, W = _layer(hk, E, H, I, 5)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, device=DEV, generator=g)
    bias = torch.randn(E, 2 * I, device=DEV, generator=g)
    got, want = bias.clone(), bias.clone()
    got[:, [3, 77, I + 9, I + 100]] = float("nan")
    want[:, [3, 77]], want[:, [I + 9, I + 100]] = 1e30, -1e30
    ys = [_run(hk, x, logits, W, H, I, E, "mxfp4", activation="swiglu_oai", bias13=b) for b in (got, want)]
    assert torch.isfinite(ys[0].float()).all()
    assert torch.equal(ys[0].view(torch.int16), ys[1].view(torch.int16))
