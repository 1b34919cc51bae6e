"""One expert's e4m3 NaN codes do not reach another expert's tokens: the partial sums of an item's last fragment are still in
registers when the next item starts. Experts of few rows whose weights hold NaN come in front of experts whose rows fill the
last fragment of an item; the latter's tokens have to be, bit for bit, what they are beside clean weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("long", [144, 288])   # items of 144 rows, and of 288
def test_nan_weights_of_an_expert_of_few_rows(hk, long):
    print(f"fp8blk expert isolation long={long}", flush=True)
    # numbers of K-steps that are multiples of four (the streaming kernel walks K-steps of zeros behind others); several items
    # a workgroup in both GEMMs, whose next item is the 32nd behind: 24 and 6 items for three experts
    H, I, E = 512, 1024, 258
    rows = [10, long, long] * (E // 3)
    T = sum(rows)
    g = torch.Generator(device=DEV).manual_seed(long)
    e4m3 = lambda *s: (torch.randn(*s, device=DEV, generator=g) * 40).to(torch.float8_e4m3fn)
    scales = lambda *s: torch.exp2(torch.randint(-12, -4, s, device=DEV, generator=g).float())
    x, w13, w2 = e4m3(T, H), e4m3(E, 2 * I, H), e4m3(E, H, I)
    xs, s13, s2 = scales(T, H // 128), scales(E, 2 * I // 128, H // 128), scales(E, H // 128, I // 128)
    ids = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(rows, device=DEV))
    ids = ids[torch.randperm(T, device=DEV, generator=g)]
    logits = torch.full((T, E), -30.0, device=DEV)
    logits[torch.arange(T, device=DEV), ids] = 30.0
    ws = torch.empty(hk.tk_kernel.moe_fp8blk_workspace_bytes(T, H, I, E, 1), dtype=torch.uint8, device=DEV)
    assert hk.load_library().hk_moe_fp8blk_item_rows(T, H, I, E, 1) == long

    def run(a, b):
        W = hk.tk_kernel.MoeFp8BlkShuffledWeights.from_plain(a, s13, b, s2)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=DEV)
        hk.tk_kernel.dispatch_moe_fp8blk(x, xs, logits, None, W, None, None, None, y, 1, 1, 1, 1.0, ws)
        torch.cuda.synchronize()
        return y

    def spoiled(w):
        w = w.clone()
        w.view(torch.uint8)[::3, :, -1] = 0x7F   # every row's last K-step
        return w

    clean, many = run(w13, w2), ids % 3 != 0
    assert torch.isfinite(clean.float()).all()
    for a, b in ((spoiled(w13), w2), (w13, spoiled(w2))):   # NaN in the gate+up projection, in the down projection
        y = run(a, b)
        assert not torch.equal(y[~many].view(torch.int16), clean[~many].view(torch.int16))   # it does arrive in its own tokens
        wrong = (y[many].view(torch.int16) != clean[many].view(torch.int16)).any(dim=1).sum().item()
        assert wrong == 0, f"{wrong} of {int(many.sum())} tokens of experts with clean weights"
