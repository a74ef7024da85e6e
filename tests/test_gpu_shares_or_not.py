"""A loss's recursion on both sides of the lines from which it passes shares instead of p (one, two, three and four
bands of rows, in workgroups of their own and together), against the recursion's own node, which always passes shares,
on the same log-probabilities: the same bits."""
import pytest
import torch

import fast_rnnt_amd as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["regular", "modified"])
@pytest.mark.parametrize("B,S,T", [(3, 20, 30), (3, 63, 199), (3, 64, 199), (3, 64, 200), (2, 127, 199), (2, 127, 200),
                                   (2, 128, 119), (2, 128, 120), (2, 200, 119), (2, 200, 120), (100, 130, 399),
                                   (100, 130, 400), (2, 300, 399), (2, 300, 400)])
def test_both_sides_of_the_lines(gpu_device, B, S, T, kind):
    g = torch.Generator().manual_seed(S + T)
    C = 7
    lm, am = (torch.randn(B, n, C, generator=g).to(gpu_device) for n in (S + 1, T))
    sym = torch.randint(0, C, (B, S), generator=g).to(gpu_device)
    t_end = torch.randint(T // 2, T + 1, (B,), generator=g)
    s_end = torch.minimum(torch.randint(S // 2, S + 1, (B,), generator=g), t_end)
    zero = torch.zeros_like(t_end)
    boundary = torch.stack([zero, zero, s_end, t_end], 1).to(gpu_device)
    loss, (gx, gy) = F.rnnt_loss_simple(lm, am, sym, 0, boundary=boundary, rnnt_type=kind, reduction="none",
                                        return_grad=True)
    px, py = F.get_rnnt_logprobs(lm, am, sym, 0, boundary=boundary, rnnt_type=kind)
    px, py = px.detach().requires_grad_(), py.detach().requires_grad_()
    scores = F.mutual_information_recursion(px, py, boundary)
    want = torch.autograd.grad(scores.sum(), (px, py))
    assert torch.equal(loss, -scores.detach())
    for a, b in zip((gx, gy), want):
        assert torch.equal(a, b)
