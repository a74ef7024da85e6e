"""Where an autograd node stands in for torch operations: what passes through them -- a second
derivative, a tangent, a write to a view -- passes through it as well."""
import pytest
import torch
import torch.autograd.forward_ad as fwd

import fast_rnnt_amd

pytestmark = pytest.mark.gpu


def _pruning_inputs(device, R=3, dtype=torch.float64):
    g = torch.Generator().manual_seed(7)
    B, T, S, C = 2, 6, 5, 4
    am = torch.randn(B, T, C, generator=g, dtype=dtype).to(device).requires_grad_(True)
    lm = torch.randn(B, S + 1, C, generator=g, dtype=dtype).to(device).requires_grad_(True)
    begin = torch.tensor([[0, 0, 1, 2, 2, 3], [0, 1, 1, 1, 3, 3]])
    return am, lm, (begin.unsqueeze(2) + torch.arange(R)).to(device)


@pytest.mark.parametrize("R", [1, 3])
def test_second_derivatives_of_the_pruning(gpu_device, R):
    am, lm, ranges = _pruning_inputs(gpu_device, R)
    prune = fast_rnnt_amd.do_rnnt_pruning
    assert torch.autograd.gradgradcheck(lambda a, l: prune(a, l, ranges), (am, lm))
    assert torch.autograd.gradgradcheck(lambda a: prune(a, lm, ranges)[0], (am,))
    assert torch.autograd.gradgradcheck(lambda l: prune(am.detach(), l, ranges)[1], (lm,))
    # a gradient penalty, against the same with torch's own operations
    rows = ranges.reshape(2, -1, 1).expand(2, 6 * R, 4)
    want, got = [], []
    for out, kept in ((want, (am.unsqueeze(2).expand(2, 6, R, 4),
                              torch.gather(lm, 1, rows).reshape(2, 6, R, 4))),
                      (got, prune(am, lm, ranges))):
        grads = torch.autograd.grad(torch.tanh(kept[0] + kept[1]).sum(), (am, lm), create_graph=True)
        out.extend(torch.autograd.grad(sum(x.square().sum() for x in grads), (am, lm)))
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-12, atol=1e-12)


def test_a_tangent_of_am_passes_through_the_pruning(gpu_device):
    am, lm, ranges = _pruning_inputs(gpu_device)
    tangent = torch.randn_like(am)
    with fwd.dual_level():
        am_pruned, lm_pruned = fast_rnnt_amd.do_rnnt_pruning(fwd.make_dual(am, tangent), lm, ranges)
        got = fwd.unpack_dual(am_pruned).tangent
        assert torch.equal(got, tangent.unsqueeze(2).expand(am_pruned.shape))
        assert lm_pruned.requires_grad and am_pruned.requires_grad


def test_one_kept_position_may_be_written_to(gpu_device):
    am, lm, ranges = _pruning_inputs(gpu_device, R=1)
    am_pruned, lm_pruned = fast_rnnt_amd.do_rnnt_pruning(am * 1, lm, ranges)
    am_pruned.mul_(2)
    (am_pruned + lm_pruned).sum().backward()
    assert torch.equal(am.grad, torch.full_like(am, 2.0))


@pytest.mark.parametrize("R", [1, 3])
def test_am_may_be_written_to_after_the_pruning(gpu_device, R):
    am, lm, ranges = _pruning_inputs(gpu_device, R)
    weights = torch.randn(2, 6, R, 4, dtype=am.dtype, device=gpu_device)
    # a parameter that is updated in between
    am_pruned, lm_pruned = fast_rnnt_amd.do_rnnt_pruning(am, lm, ranges)
    with torch.no_grad():
        am.add_(1)
    assert torch.equal(am_pruned, am.unsqueeze(2).expand(2, 6, R, 4))
    (weights * (am_pruned + lm_pruned)).sum().backward()
    assert torch.allclose(am.grad, weights.sum(2), rtol=1e-12, atol=1e-12)
    # an activation that is changed on record: what am_pruned shows of it is differentiated too
    results = []
    for prune in (True, False):
        x, y = am.detach().clone().requires_grad_(True), lm.detach().clone().requires_grad_(True)
        hidden = x * 3
        if prune:
            kept = fast_rnnt_amd.do_rnnt_pruning(hidden, y, ranges)
        else:
            rows = ranges.reshape(2, -1, 1).expand(2, 6 * R, 4)
            kept = (hidden.unsqueeze(2).expand(2, 6, R, 4),
                    torch.gather(y, 1, rows).reshape(2, 6, R, 4))
        hidden.mul_(2)
        kept[1].add_(kept[0])  # a joiner that adds in place
        (weights * torch.tanh(kept[1])).sum().backward()
        results.append((x.grad, y.grad))
    for a, b in zip(*results):
        assert torch.allclose(a, b, rtol=1e-12, atol=1e-12)
    # a tensor that a later operation has kept: refused, as with torch's own view
    hidden = am * 1
    am_pruned, lm_pruned = fast_rnnt_amd.do_rnnt_pruning(hidden, lm, ranges)
    out = (am_pruned * lm_pruned).sum()
    hidden.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_gradients_of_the_recursion_keep_the_history_of_the_scores_gradient(gpu_device, dtype):
    g = torch.Generator().manual_seed(3)
    B, S, T = 3, 4, 6
    px = torch.randn(B, S, T + 1, generator=g, dtype=dtype).to(gpu_device).requires_grad_(True)
    py = torch.randn(B, S + 1, T, generator=g, dtype=dtype).to(gpu_device).requires_grad_(True)
    weights = torch.tensor([1.0, 2.0, -0.5], dtype=dtype, device=gpu_device, requires_grad=True)
    scores, occupation = fast_rnnt_amd.mutual_information_recursion(px, py, return_grad=True)
    occ_x, occ_y = (x.clone() for x in occupation)
    gx, gy = torch.autograd.grad((weights * scores).sum(), (px, py), create_graph=True)
    for got, occ, handed_out in ((gx, occ_x, occupation[0]), (gy, occ_y, occupation[1])):
        assert torch.equal(handed_out.detach(), got.detach())  # (scaled in place)
        assert torch.equal(got.detach(), occ * weights.detach().reshape(B, 1, 1))
    (gx.sum() + gy.square().sum()).backward()
    want = occ_x.sum((1, 2)) + 2 * weights.detach() * occ_y.square().sum((1, 2))
    assert torch.allclose(weights.grad, want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("return_grad", [False, True])
@pytest.mark.parametrize("path", ["simple", "smoothed", "smoothed_constrained", "joint"])
def test_a_second_backward_is_right_or_refused(gpu_device, path, return_grad):
    g = torch.Generator().manual_seed(4)
    B, S, T, C = 2, 4, 7, 5
    symbols = torch.randint(1, C, (B, S), generator=g).to(gpu_device)
    if path == "joint":
        leaves = [torch.randn(B, T, S + 1, C, generator=g)]
    else:
        leaves = [torch.randn(B, S + 1, C, generator=g), torch.randn(B, T, C, generator=g)]
    leaves = [x.to(gpu_device).requires_grad_(True) for x in leaves]
    kind = "constrained" if path == "smoothed_constrained" else "regular"
    loss_fn = {"simple": fast_rnnt_amd.rnnt_loss_simple, "joint": fast_rnnt_amd.rnnt_loss,
               "smoothed": fast_rnnt_amd.rnnt_loss_smoothed,
               "smoothed_constrained": fast_rnnt_amd.rnnt_loss_smoothed}[path]
    loss = loss_fn(*leaves, symbols, 0, rnnt_type=kind, reduction="mean", return_grad=return_grad)
    loss = loss[0] if return_grad else loss
    first = torch.autograd.grad(loss, leaves, retain_graph=True)
    if path == "joint" and not return_grad:  # (nothing is scaled in place)
        assert all(torch.equal(a, b) for a, b in zip(first, torch.autograd.grad(loss, leaves)))
    else:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(loss, leaves)
