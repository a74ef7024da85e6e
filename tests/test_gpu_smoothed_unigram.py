"""The gradient of the smoothed loss's unigram where the (utterance, row) pairs just fill a chunk of the kernel that
sums them per symbol, fall short of it, or leave one for the next.  Oracle: the CPU restatement in float32."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S", [(1, 1), (3, 20), (63, 64), (64, 63), (241, 16), (512, 7), (745, 10)])
def test_pairs_at_the_edges_of_chunks(gpu_device, B, S):
    T, C, term = 12, 18, 17
    g = torch.Generator().manual_seed(B)
    symbols = torch.randint(0, C, (B, S), generator=g)
    lm, am = torch.randn(B, S + 1, C, generator=g), torch.randn(B, T, C, generator=g)
    zero = torch.zeros(B, dtype=torch.int64)
    s_end = torch.randint(1, min(S, T) + 1, (B,), generator=g)
    boundary = torch.stack([zero, zero, s_end, zero + T], 1)
    args = dict(lm_only_scale=0.1, am_only_scale=0.3, reduction="sum")
    cpu = [x.clone().requires_grad_(True) for x in (lm, am)]
    gpu = [x.to(gpu_device).requires_grad_(True) for x in (lm, am)]
    O.loss_smoothed(*cpu, symbols, term, boundary=boundary, **args).backward()
    fast_rnnt_amd.rnnt_loss_smoothed(*gpu, symbols.to(gpu_device), term, boundary=boundary.to(gpu_device),
                                     **args).backward()
    for x, y in zip(gpu, cpu):
        off = (x.grad.cpu() - y.grad).abs()
        # (the tolerance of the gradients at other sizes; the unigram's terms are means over the rows)
        assert bool((off <= 2e-4 + 1e-4 * y.grad.abs()).all()), off.max().item()
