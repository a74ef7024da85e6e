"""The loss of a call without a gradient, which the recursion's forward kernel forms of the scores itself,
against the one that the backward kernel forms: the same sums in the same order."""
import pytest
import torch

import fast_rnnt_amd as F

pytestmark = pytest.mark.gpu


# one utterance, a wave's lanes all but one, one and two to a lane; one band of rows and two, and bands of
# which some utterances leave the second empty
@pytest.mark.parametrize("reduction", ["none", "mean", "sum"])
@pytest.mark.parametrize("rnnt_type", ["regular", "modified", "constrained"])
@pytest.mark.parametrize("B,S,T,C", [(1, 5, 9, 11), (63, 3, 8, 16), (65, 4, 9, 8), (130, 2, 7, 12), (3, 70, 90, 8)])
def test_same_loss_with_and_without_a_gradient(B, S, T, C, rnnt_type, reduction):
    g = torch.Generator().manual_seed(B + S)
    t_end = torch.randint(max(S, T // 2), T + 1, (B,), generator=g)
    s_end = torch.randint(1, S + 1, (B,), generator=g)
    zero = torch.zeros(B, dtype=torch.int64)
    bnd = torch.stack([zero, zero, s_end, t_end], dim=1).cuda()
    sym = torch.randint(1, C, (B, S), generator=g).cuda()
    logits = torch.randn(B, T, S + 1, C, generator=g).cuda()
    am, lm = torch.randn(B, T, C, generator=g).cuda(), torch.randn(B, S + 1, C, generator=g).cuda()
    for boundary in (bnd, None):
        kinds = dict(boundary=boundary, rnnt_type=rnnt_type, reduction=reduction)
        for _ in range(2):
            with torch.no_grad():
                got = F.rnnt_loss(logits, sym, 0, **kinds)
                simple = F.rnnt_loss_simple(lm, am, sym, 0, **kinds)
            want = F.rnnt_loss(logits.clone().requires_grad_(), sym, 0, **kinds).detach()
            simple_want = F.rnnt_loss_simple(lm.clone().requires_grad_(), am, sym, 0, **kinds).detach()
            assert torch.isfinite(got).all() and torch.equal(got, want)
            assert torch.equal(simple, simple_want)
