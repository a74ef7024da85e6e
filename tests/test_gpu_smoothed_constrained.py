"""rnnt_loss_smoothed of the constrained lattice, in one node as the other lattices' (the row below joins px, and
its gradient comes back there): sizes at the edges of tiles, windows, the delay penalty, with and without
occupation gradients handed out and an am-only model.  Oracle: the CPU restatement in float32."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,T,C", [(1, 1, 1, 1), (2, 3, 9, 5), (2, 31, 33, 64), (1, 64, 128, 65),
                                     (3, 100, 129, 300), (2, 32, 64, 1000), (30, 20, 70, 130)])
def test_constrained_smoothed_loss(gpu_device, B, S, T, C):
    g = torch.Generator().manual_seed(B + S + T + C)
    t_end = (T * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1)
    s_end = torch.minimum((S * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1), t_end)
    t_end[0], s_end[0] = T, min(S, T)
    zero = torch.zeros_like(t_end)
    windows = torch.stack([zero, zero, s_end, t_end], 1)
    symbols = torch.randint(0, C, (B, S), generator=g)
    lm, am = torch.randn(B, S + 1, C, generator=g), torch.randn(B, T, C, generator=g)
    weights = 1 + torch.rand(B, generator=g)
    for term, l, a, handed_out in [(0, 0.25, 0.0, True), (C - 1, 0.1, 0.2, False)]:
        for boundary in (windows, None):
            cpu = [x.clone().requires_grad_(True) for x in (lm, am)]
            gpu = [x.to(gpu_device).requires_grad_(True) for x in (lm, am)]
            args = dict(lm_only_scale=l, am_only_scale=a, rnnt_type="constrained", delay_penalty=0.01,
                        reduction="none")
            want = O.loss_smoothed(*cpu, symbols, term, boundary=boundary, **args)
            bnd = None if boundary is None else boundary.to(gpu_device)
            got = fast_rnnt_amd.rnnt_loss_smoothed(*gpu, symbols.to(gpu_device), term, boundary=bnd,
                                                   return_grad=handed_out, **args)
            got = got[0] if handed_out else got
            # (a score is a sum of S + T values that round a few times each)
            bound = 8 * (S + T) * 2.0 ** -24 * want.detach().abs().clamp(min=1)
            assert bool(((got.detach().cpu() - want.detach()).abs() <= bound).all())
            (weights * want).sum().backward()
            (weights.to(gpu_device) * got).sum().backward()
            for x, y in zip(gpu, cpu):
                off = (x.grad.cpu() - y.grad).abs()
                # (the tolerance of the other lattices' gradients, whose bf16-split products these are)
                assert bool((off <= 2e-4 + 1e-4 * y.grad.abs()).all()), off.max().item()


@pytest.mark.parametrize("am_scale", [0.0, 0.1])
def test_boundary_written_to_between_forward_and_backward(gpu_device, am_scale):
    """The gradients are those of the rows that the loss was formed with: a program may fill one boundary buffer for one
    batch after the other."""
    B, S, T, C = 5, 20, 70, 33
    g = torch.Generator().manual_seed(0)
    lm, am = (torch.randn(B, n, C, generator=g).to(gpu_device).requires_grad_() for n in (S + 1, T))
    symbols = torch.randint(0, C, (B, S), generator=g).to(gpu_device)
    one, two = (torch.tensor([[0, 0, s, t]] * B).to(gpu_device) for s, t in ((S, T), (S - 7, T - 30)))

    def loss(boundary):
        return fast_rnnt_amd.rnnt_loss_smoothed(lm, am, symbols, 0, 0.25, am_scale, boundary=boundary,
                                                rnnt_type="constrained", reduction="sum")

    want = [torch.autograd.grad(loss(rows.clone()), (lm, am)) for rows in (one, two)]
    buffer = one.clone()
    first = loss(buffer)
    buffer.copy_(two)
    second = loss(buffer)
    buffer.zero_()
    for value, grads in ((second, want[1]), (first, want[0])):
        for a, b in zip(torch.autograd.grad(value, (lm, am)), grads):
            assert torch.equal(a, b)
