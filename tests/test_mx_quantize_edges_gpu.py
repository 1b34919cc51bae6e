"""MX quantization where its kernels change form: rows per thread (large inputs, a last group of one to three rows), and the
positions of a token block's slots held by the lanes of a wave (up to eight choices a token) or looked up one by one."""
import numpy as np
import pytest
import torch

from oracle import formats as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("cols", [96, 2880])
@pytest.mark.parametrize("rows", [1, 1023, 2730, 4096, 4097, 4098, 4099, 32771])
def test_rows_of_every_remainder(hk, rows, cols, fmt):
    rng = np.random.default_rng(rows + cols)
    x = F.bf16_to_f32(F.bf16_round(rng.standard_normal((rows, cols)).astype(np.float32)))
    xt = torch.from_numpy(x).to(DEV).to(torch.bfloat16)
    pitch, width = -(-cols // 256) * 8, cols if fmt == "mxfp8" else cols // 2
    guard = 64
    packed = torch.full((rows * width + guard,), 0xAA, dtype=torch.uint8, device=DEV)
    scales = torch.full((rows * pitch + guard,), 0xAA, dtype=torch.uint8, device=DEV)
    out = packed[:rows * width].view(rows, width), scales[:rows * pitch].view(rows, pitch)
    if fmt == "mxfp8":
        hk.tk_kernel.dispatch_mxfp8_quantize_rows(xt, out[0].view(torch.float8_e4m3fn), out[1])
        want_p, want_s = F.quantize_mxfp8(x)
    else:
        hk.tk_kernel.dispatch_mxfp4_quantize_rows(xt, *out)
        want_p, want_s = F.quantize_mxfp4(x)
    torch.cuda.synchronize()
    assert np.array_equal(out[0].cpu().numpy(), want_p)
    got = out[1].cpu().numpy()
    assert np.array_equal(got[:, :cols // 32], want_s) and (got[:, cols // 32:] == 127).all()
    assert (packed[-guard:] == 0xAA).all() and (scales[-guard:] == 0xAA).all()


@pytest.mark.parametrize("act_format", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 12])
def test_positions_of_any_number_of_choices(hk, k, act_format):
    """Permuting quantization (biases) against the gathering one (bias of zeros left out): the same layer, bit for bit."""
    T, E, H, I = 403, 16, 288, 160
    g = torch.Generator(device=DEV).manual_seed(k)
    w13 = hk.quant.quantize_mxfp4(torch.randn(E, 2 * I, H, device=DEV, generator=g) * 0.2)
    w2 = hk.quant.quantize_mxfp4(torch.randn(E, H, I, device=DEV, generator=g) * 0.2)
    W = hk.tk_kernel.MoeMxfp4ShuffledWeights.from_plain(w13[0], hk.quant.pad_scales(w13[1]), w2[0], hk.quant.pad_scales(w2[1]))
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, device=DEV, generator=g)
    ys = []
    for options in ({}, {"bias13": torch.zeros(E, 2 * I, device=DEV)}):
        ws = torch.empty(hk.tk_kernel.moe_mxfp4_workspace_bytes(T, H, I, E, k, act_format), dtype=torch.uint8, device=DEV)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_mxfp4(x, logits, W, None, None, None, y, k, ws, act_format=act_format, **options)
        torch.cuda.synchronize()
        ys.append(y)
    assert torch.isfinite(ys[0].float()).all()
    assert torch.equal(ys[0].view(torch.int16), ys[1].view(torch.int16))
