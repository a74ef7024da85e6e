"""The recursion's backward operator with gradients of the scores that are not finite: they reach the cells of their own
utterance's window that a gradient reaches at all, as in the oracle, and nothing else."""
import math

import pytest
import torch

from fast_rnnt_amd import _fast_rnnt
from oracle import recursion as oracle

pytestmark = pytest.mark.gpu


# one band of rows, several together (float64: always) and apart, more than four
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T", [(1, 1), (20, 45), (63, 64), (100, 130), (130, 1200), (300, 320)])
def test_seeds_that_are_not_finite(gpu_device, S, T, modified, dtype):
    g = torch.Generator().manual_seed(S + T)
    seeds = torch.tensor([1.0, math.nan, math.inf, math.nan, -0.5, -math.inf, math.nan], dtype=dtype)
    rows = torch.tensor([[0, 0, S, T], [S // 3, T // 4, S, T - T // 5], [0, T // 3, S - S // 4, T], [0, 0, S // 2, T],
                         [0, 0, S, T], [S // 2, 0, S, T], [0, T, S, T]])
    B = len(rows)
    px = (-1 + torch.randn(B, S, T if modified else T + 1, generator=g)).to(dtype)
    py = (-1 + torch.randn(B, S + 1, T, generator=g)).to(dtype)
    p = torch.zeros(B, S + 1, T + 1, dtype=dtype)
    oracle.mi_forward(px, py, rows, p)
    want = oracle.mi_backward(px, py, rows, p, seeds)
    ones = oracle.mi_backward(px, py, rows, p, torch.ones_like(seeds))
    got = _fast_rnnt.mutual_information_backward(*(x.to(gpu_device) for x in (px, py, rows, p)), seeds.to(gpu_device))
    for h, w, one in zip(got, want, ones):
        h = h.cpu()
        # the same operations on the same p: an ulp of exp per cell and a rounding per step of a path
        scale = (S + T) * torch.finfo(dtype).eps
        for b in range(B):
            if math.isfinite(seeds[b]):
                assert torch.allclose(h[b], w[b], rtol=8 * scale, atol=8 * scale)
            elif math.isnan(seeds[b]):
                assert torch.equal(torch.isnan(h[b]), torch.isnan(w[b]))
                assert not h[b][~torch.isnan(w[b])].any()
            s0, t0, s1, t1 = rows[b].tolist()
            inside = torch.zeros_like(h[b], dtype=torch.bool)
            inside[s0:s1 + 1, t0:t1 + 1] = True
            assert not h[b][~inside].any()
            assert one[b][~inside].eq(0).all()
