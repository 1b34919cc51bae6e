"""The un-permute shares a token's columns among workgroups for small batches: widths around a workgroup's column
chunk (512), token counts on both sides of the rule, every form of the choice count."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (1, 4, 504), (3, 4, 512), (4, 4, 520), (4, 4, 2880), (16, 8, 7168),
                                   (2, 10, 1032), (255, 2, 576), (256, 2, 576), (257, 3, 2056)])
@pytest.mark.parametrize("with_add", [False, True])
def test_every_column_is_written_once(hk, T, k, H, with_add):
    """Small integers: add + sum_j w_j o_j stays below 256 in magnitude, so fp32 and bf16 hold it exactly."""
    rng = np.random.default_rng(T * 10007 + H)
    o = rng.integers(-8, 9, size=(T * k, H)).astype(np.float32)
    w = rng.integers(1, 4, size=(T, k)).astype(np.float32)   # 10 choices: at most 8 * 3 * 10 + 8 = 248
    inv = rng.permutation(T * k).astype(np.int32)
    add = rng.integers(-8, 9, size=(T, H)).astype(np.float32)
    want = add.copy() if with_add else np.zeros((T, H), dtype=np.float32)
    for j in range(k):
        want += w[:, j:j + 1] * o[inv[np.arange(T) * k + j]]
    bf = lambda a: torch.from_numpy(a).to(DEV).to(torch.bfloat16)
    y = torch.full((T + 1, H), 777.0, dtype=torch.bfloat16, device=DEV)
    hk.tk_kernel.dispatch_moe_unpermute(bf(o), torch.from_numpy(w).to(DEV), torch.from_numpy(inv).to(DEV), y[:T],
                                        add=bf(add) if with_add else None)
    torch.cuda.synchronize()
    assert np.array_equal(y[:T].float().cpu().numpy(), want)
    assert torch.all(y[T] == y.new_tensor(777.0))   # the row behind the last token
