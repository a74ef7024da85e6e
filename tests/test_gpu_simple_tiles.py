"""rnnt_loss_simple where the kernels' choice of tiles and their splits into chunks can go wrong:
sizes on either side of a tile of lattice rows, frames and vocabulary entries, sums over few and
many chunks, batches small and large, 2-byte inputs, long lists of equal symbols.  Oracle: the CPU
restatement on the same values in float32."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu
# (B, S, T, C)
SIZES = [(1, 1, 1, 1), (2, 1, 3, 31), (1, 31, 33, 32), (2, 32, 64, 33), (3, 63, 65, 64),
         (1, 64, 64, 65), (2, 95, 96, 129), (1, 127, 129, 300), (2, 128, 140, 70),
         (1, 20, 40, 4097), (2, 60, 70, 2600), (1, 130, 260, 1700), (5, 100, 190, 2050),
         (40, 70, 300, 40), (70, 33, 130, 130), (30, 130, 280, 66)]


@pytest.mark.parametrize("B,S,T,C", SIZES)
def test_simple_loss_at_the_edges_of_tiles(gpu_device, B, S, T, C):
    g = torch.Generator().manual_seed(B + S + T + C)
    t_end = (T * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1)
    s_end = torch.minimum((S * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1), t_end)
    t_end[0], s_end[0] = T, min(S, T)
    zero = torch.zeros_like(t_end)
    boundary = torch.stack([zero, zero, s_end, t_end], 1)
    symbols = torch.randint(0, C, (B, S), generator=g)
    symbols[0] = C // 2  # every lattice row of an utterance on one vocabulary entry
    for dtype, kind in [(torch.float32, "regular"), (torch.bfloat16, "modified"),
                        (torch.float16, "constrained")]:
        print(f"B={B} S={S} T={T} C={C} {dtype} {kind}", flush=True)
        lm = (2 * torch.randn(B, S + 1, C, generator=g)).to(dtype)
        am = (2 * torch.randn(B, T, C, generator=g)).to(dtype)
        cpu = [x.float().clone().requires_grad_(True) for x in (lm, am)]
        gpu = [x.to(gpu_device).requires_grad_(True) for x in (lm, am)]
        args = dict(rnnt_type=kind, delay_penalty=0.01, reduction="mean")
        want = O.loss_simple(*cpu, symbols, 0, boundary=boundary, **args)
        got, occupation = fast_rnnt_amd.rnnt_loss_simple(
            *gpu, symbols.to(gpu_device), 0, boundary=boundary.to(gpu_device), return_grad=True,
            **args)
        assert abs(got.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
        (3.0 * want).backward()
        (3.0 * got).backward()
        assert occupation[0].dtype == torch.float32
        ulp = {torch.float32: 1e-4, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
        for x, y in zip(gpu, cpu):
            assert x.grad.dtype == dtype
            off = (x.grad.float().cpu() - y.grad).abs()
            assert bool((off <= 2e-4 + ulp * y.grad.abs()).all()), off.max().item()
