"""Layers whose experts get only a few rows (decode steps, small batches) run the few-rows grouped GEMM on the
pre-shuffled weights: against the oracle, and bit for bit against the plain layout's kernel, at the edges of its
row fragments, column groups and K-steps."""
import numpy as np
import pytest
import torch

from oracle import formats as F
from oracle import gemm as G
from oracle import moe as O

DEV = "cuda:0"
TOL = 1e-2   # as for the layer's other tests


def _bf16(a):
    return F.bf16_to_f32(F.bf16_round(np.asarray(a, dtype=np.float32)))


def _to_bf16_tensor(a):
    return torch.from_numpy(F.bf16_round(a).view(np.int16)).view(torch.bfloat16).to(DEV)


def _logits(rng, T, E, hot):
    """`hot` of the tokens prefer expert 1: more rows than one work item holds."""
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:hot, 1] += 20.0
    return logits


# rows of the hot expert around 16 and 32 (one and two row fragments), few and many experts; I and H with partial
# column groups (32, 96, 160), K tails of one MX block, one K-step, exact K-steps and more K-steps than the ring
MXFP4 = [
    # T, E, k, H, I, hot
    (1, 4, 2, 256, 128, 0),
    (1, 2, 1, 32, 32, 0),
    (15, 16, 2, 288, 96, 15),
    (16, 16, 2, 512, 160, 16),
    (17, 32, 4, 544, 352, 17),
    (33, 64, 4, 1056, 256, 33),
    (40, 24, 4, 800, 288, 31),     # mean above 4 rows: two fragments
    (64, 33, 4, 2880, 320, 33),
    (64, 33, 4, 256, 1312, 64),
]


@pytest.mark.gpu
@pytest.mark.parametrize("ext", [False, True])
@pytest.mark.parametrize("act", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("T,E,k,H,I,hot", MXFP4)
def test_moe_mxfp4_few_rows(hk, T, E, k, H, I, hot, act, ext):
    print(f"moe_mxfp4 few rows T={T} E={E} k={k} H={H} I={I} hot={hot} {act} ext={ext}", flush=True)
    # MXFP8 layers with a mean above 4 rows take the streaming kernel
    rows = 16 if T * k <= 4 * E else 0 if act == "mxfp8" else 32
    assert hk.load_library().hk_moe_mxfp4_few_rows(T, H, I, E, k, act == "mxfp8", ext) == rows
    rng = np.random.default_rng(T + E + H + I)
    x = _bf16(rng.standard_normal((T, H)))
    logits = _logits(rng, T, E, hot)
    w13p, w13s = F.quantize_mxfp4((rng.standard_normal((E, 2 * I, H)) * 0.2).astype(np.float32))
    w2p, w2s = F.quantize_mxfp4((rng.standard_normal((E, H, I)) * 0.2).astype(np.float32))
    bias = dict(bias13=rng.standard_normal((E, 2 * I)).astype(np.float32),
                bias2=rng.standard_normal((E, H)).astype(np.float32)) if ext else {}
    dev = lambda a: torch.from_numpy(a).to(DEV)
    opts = {n: dev(b) for n, b in bias.items()}
    if ext:
        opts["activation"] = "swiglu_oai"
    plain = [dev(w13p), hk.quant.pad_scales(dev(w13s)), dev(w2p), hk.quant.pad_scales(dev(w2s))]
    W = hk.tk_kernel.MoeMxfp4ShuffledWeights.from_plain(*plain)
    # whatever a workspace holds before the call, NaN scales among it, reaches no result
    ws = torch.full((hk.tk_kernel.moe_mxfp4_workspace_bytes(T, H, I, E, k, act_format=act),), 255, dtype=torch.uint8, device=DEV)
    xt, lt = _to_bf16_tensor(x), dev(logits)
    guard = 64   # rows behind y that nothing may touch
    y = torch.full((T + guard, H), 7.0, dtype=torch.bfloat16, device=DEV)
    hk.tk_kernel.dispatch_moe_mxfp4(xt, lt, W, None, None, None, y[:T], k, ws, act_format=act, **opts)
    torch.cuda.synchronize()
    assert (y[T:] == 7.0).all()
    got = y[:T].float().cpu().numpy()
    ids, w = O.topk_softmax(logits, k)
    want = F.bf16_to_f32(O.moe_mxfp4_forward(x, ids, w, w13p, w13s, w2p, w2s, act_format=act,
                                             activation="swiglu_oai" if ext else "silu", **bias)[0])
    err = G.rel_fro_error(got, want)
    assert np.isfinite(got).all() and err <= TOL, err
    if act == "mxfp4":
        yp = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_mxfp4(xt, lt, *plain, yp, k, ws, **opts)
        torch.cuda.synchronize()
        assert torch.equal(yp.view(torch.int16), y[:T].view(torch.int16))
