"""rnnt_loss_smoothed's fused forward and backward at the sizes where the smoothing terms inside the
gradient products can go wrong: tile edges, repeated symbols, the termination symbol anywhere,
windows, the delay penalty, with and without occupation gradients handed out.  Oracle: the CPU
restatement in float32."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["regular", "modified"])
@pytest.mark.parametrize("B,S,T,C", [(1, 1, 1, 1), (2, 3, 9, 5), (2, 63, 65, 64), (1, 64, 128, 65),
                                     (3, 100, 129, 300), (2, 130, 260, 70), (30, 20, 70, 130)])
def test_smoothed_loss_at_the_edges_of_tiles(gpu_device, B, S, T, C, kind):
    g = torch.Generator().manual_seed(B + S + T + C)
    t_end = (T * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1)
    s_end = torch.minimum((S * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1), t_end)
    t_end[0], s_end[0] = T, min(S, T)
    zero = torch.zeros_like(t_end)
    windows = torch.stack([zero, zero, s_end, t_end], 1)
    symbols = torch.randint(0, C, (B, S), generator=g)
    symbols[0] = C // 2
    lm, am = torch.randn(B, S + 1, C, generator=g), torch.randn(B, T, C, generator=g)
    for term, l, a, handed_out in [(0, 0.25, 0.0, True), (C - 1, 0.1, 0.2, False)]:
        for boundary in (windows, None) if S <= T else (windows,):
            print(f"B={B} S={S} T={T} C={C} {kind} term={term}", flush=True)
            cpu = [x.clone().requires_grad_(True) for x in (lm, am)]
            gpu = [x.to(gpu_device).requires_grad_(True) for x in (lm, am)]
            args = dict(lm_only_scale=l, am_only_scale=a, rnnt_type=kind, delay_penalty=0.01,
                        reduction="mean")
            want = O.loss_smoothed(*cpu, symbols, term, boundary=boundary, **args)
            bnd = None if boundary is None else boundary.to(gpu_device)
            got = fast_rnnt_amd.rnnt_loss_smoothed(*gpu, symbols.to(gpu_device), term, boundary=bnd,
                                                   return_grad=handed_out, **args)
            got = got[0] if handed_out else got
            assert abs(got.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
            (3.0 * want).backward()
            (3.0 * got).backward()
            for x, y in zip(gpu, cpu):
                off = (x.grad.cpu() - y.grad).abs()
                assert bool((off <= 2e-4 + 1e-4 * y.grad.abs()).all()), off.max().item()
