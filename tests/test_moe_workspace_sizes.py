"""A layer's workspace never shrinks when the batch grows: a program that allocates it once for its largest batch runs
every smaller one in it, on whichever kernels the smaller batch takes."""
import pytest
import torch

import hipkittens_amd as hk

tk = hk.tk_kernel


# H, I, E, k: the layers of the benchmark, experts that every token passes through, one choice per token, a wide hidden
# layer (more bytes per row of h in fp32 than of the down GEMM's output) and a narrow one
LAYERS = [(7168, 2048, 256, 8), (7168, 2048, 1, 1), (2048, 768, 128, 8), (1024, 512, 64, 6), (512, 4096, 8, 2),
          (7168, 512, 16, 4), (512, 2048, 1, 1), (2880 // 128 * 128, 2816, 128, 4)]


def _assert_never_shrinks(size, E, k):
    # every batch around the edges of the kernels' rules (up to 192 rows per expert), coarser steps above
    Ts = sorted(set(range(1, 600)) | {T for m in (1, 2, 4, 8, 16, 64, 144, 160, 192, 193)
                                      for T in range(max(1, m * E // k - 3), m * E // k + 4)} | set(range(600, 9000, 97)))
    sizes = [size(T) for T in Ts]
    assert all(s > 0 for s in sizes)
    shrinks = [(a, b) for a, b, s, t in zip(Ts, Ts[1:], sizes, sizes[1:]) if t < s]
    assert not shrinks, shrinks[:5]


@pytest.mark.parametrize("H,I,E,k", LAYERS)
def test_fp8blk_size_never_shrinks(H, I, E, k):
    _assert_never_shrinks(lambda T: tk.moe_fp8blk_workspace_bytes(T, H, I, E, k), E, k)


@pytest.mark.parametrize("act", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("H,I,E,k", [(2880, 2880, 128, 4), (128, 32, 512, 1), (64, 1024, 128, 1), (2880, 2880, 8, 2),
                                     (2048, 768, 128, 8), (32, 32, 64, 2)])
def test_mxfp4_size_never_shrinks(H, I, E, k, act):
    _assert_never_shrinks(lambda T: tk.moe_mxfp4_workspace_bytes(T, H, I, E, k, act_format=act), E, k)


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,E,k,largest,batches", [(256, 1920, 1, 1, 200, (192, 191, 64, 1)), (512, 256, 32, 8, 14, (8, 5, 1)),
                                                     (256, 1024, 8, 2, 300, (60, 30, 16))])
def test_fp8blk_small_batches_in_the_largest_ones_workspace(H, I, E, k, largest, batches):
    dev = "cuda:0"
    g = torch.Generator(device=dev).manual_seed(H + I)
    rn = lambda *s: torch.randn(*s, device=dev, generator=g)
    quantized = [hk.quant.quantize_fp8_blocks(rn(E, *s) * 0.1, 128, 128) for s in ((2 * I, H), (H, I))]
    W = tk.MoeFp8BlkShuffledWeights.from_plain(*quantized[0], *quantized[1])
    size = tk.moe_fp8blk_workspace_bytes(largest, H, I, E, k)
    ws = torch.empty(size + 256, dtype=torch.uint8, device=dev)
    for T in (largest, *batches):
        xq, xs = hk.quant.quantize_fp8_blocks(rn(T, H), 1, 128)
        logits = rn(T, E)
        out = []
        for w in ((W, None, None, None), (*quantized[0], *quantized[1])):   # the plain layout's kernel has the same bits
            ws.fill_(0xFF)
            y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=dev)
            tk.dispatch_moe_fp8blk(xq, xs, logits, None, *w, y, k, 1, 1, 1.0, ws[:size])
            out.append(y)
        assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
        assert torch.all(ws[size:] == 0xFF)   # nothing is written behind the workspace
