"""One expert's weights do not reach another expert's tokens: work items of different experts follow one another in the same
accumulators. Experts of few rows whose weight scales hold the e8m0 NaN (0xFF) come in front of experts of many rows; the
latter's tokens have to be, bit for bit, what they are beside clean weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows of the experts of few rows: one fragment of 16, and up to the last that leaves a shared branch's fragments without rows
SHORT = [1, 16, 17, 33, 48, 49, 64, 65, 80, 81, 96, 97, 111, 112, 5, 30]


def _weights(hk, g, E, rows, cols, short):
    packed, scales = hk.quant.quantize_mxfp4(torch.randn(E * rows, cols, device=DEV, generator=g) * 0.2)
    packed, scales = packed.view(E, rows, -1), scales.view(E, rows, -1)
    bad = scales.clone()
    for i, e in enumerate(short):
        bad[e, (5 + i) % 16::16, i % scales.shape[2]] = 0xFF   # (every 16-column fragment of the expert)
    return packed, hk.quant.pad_scales(scales), hk.quant.pad_scales(bad)


@pytest.mark.parametrize("act_format", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("options", [{}, {"bias": True}, {"activation": "swiglu_oai", "bias": True}], ids=["plain", "biases", "swiglu"])
# (plain: rows gathered by token up to 512, MXFP4 up to 1024; else permuted; MXFP4 with experts of 1000 rows: items of 288)
@pytest.mark.parametrize("H,long", [(512, 600), (1024, 600), (1024, 1000)])
def test_nan_scale_of_an_expert_of_few_rows(hk, H, long, options, act_format):
    print(f"moe expert isolation H={H} long={long} {options} {act_format}", flush=True)
    # 512 and more items of gate+up and, at H = 1024, more than 256 of down: a workgroup's next item is the 32nd behind
    I, rows = 1024, [r for s in SHORT for r in (s, long)]
    E, T = len(rows), sum(rows)
    short = list(range(0, E, 2))
    tall = hk.load_library().hk_moe_mxfp4_item_rows(T, H, I, E, 1, act_format == "mxfp8", bool(options)) == 288
    assert tall == (long == 1000 and act_format == "mxfp4")
    g = torch.Generator(device=DEV).manual_seed(H)
    p13, s13, bad13 = _weights(hk, g, E, 2 * I, H, short)
    p2, s2, bad2 = _weights(hk, g, E, H, I, short)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(rows, device=DEV))
    ids = ids[torch.randperm(T, device=DEV, generator=g)]
    logits = torch.zeros(T, E, device=DEV)
    logits[torch.arange(T, device=DEV), ids] = 30.0
    kw = {"act_format": act_format, "activation": options.get("activation", "silu")}
    if options.get("bias"):
        kw.update(bias13=torch.randn(E, 2 * I, device=DEV, generator=g), bias2=torch.randn(E, H, device=DEV, generator=g))

    def run(a, b):
        W = hk.tk_kernel.MoeMxfp4ShuffledWeights.from_plain(p13, a, p2, b)
        ws = torch.empty(hk.tk_kernel.moe_mxfp4_workspace_bytes(T, H, I, E, 1, act_format), dtype=torch.uint8, device=DEV)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_mxfp4(x, logits, W, None, None, None, y, 1, ws, **kw)
        torch.cuda.synchronize()
        return y

    clean, many = run(s13, s2), ids % 2 == 1
    assert torch.isfinite(clean.float()).all()
    for a, b in ((bad13, s2), (s13, bad2)):   # NaN in the gate+up projection, in the down projection
        y = run(a, b)
        assert not torch.equal(y[~many].view(torch.int16), clean[~many].view(torch.int16))   # it does arrive in its own tokens
        wrong = (y[many].view(torch.int16) != clean[many].view(torch.int16)).any(dim=1).sum().item()
        assert wrong == 0, f"{wrong} of {int(many.sum())} tokens of experts with clean weights"
