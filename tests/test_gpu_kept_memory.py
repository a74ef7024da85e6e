"""What a loss on logits keeps between its forward and its backward: the normalizers and the
occupation gradients, not the lattices that only the forward needs."""
import pytest
import torch

import fast_rnnt_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["joint", "pruned"])
def test_memory_kept_for_the_backward(gpu_device, path):
    B, T, S, C, R = 4, 200, 40, 30, 5
    g = torch.Generator().manual_seed(0)
    K = S + 1 if path == "joint" else R
    logits = torch.randn(B, T, K, C, generator=g).to(gpu_device).requires_grad_(True)
    symbols = torch.randint(1, C, (B, S), generator=g).to(gpu_device)
    begin = (torch.arange(T) * (S + 2 - R) // T).reshape(1, T, 1).expand(B, T, 1)
    ranges = (begin + torch.arange(R)).to(gpu_device)

    def loss():
        if path == "joint":
            return fast_rnnt_amd.rnnt_loss(logits, symbols, 0, reduction="sum")
        return fast_rnnt_amd.rnnt_loss_pruned(logits, symbols, ranges, 0, reduction="sum")

    loss().backward()
    before = torch.cuda.memory_allocated()
    kept = loss()
    norm, px_grad, py_grad = B * T * K, B * S * (T + 1), B * (S + 1) * T
    # (the allocator hands out multiples of 512 bytes)
    assert torch.cuda.memory_allocated() - before <= 4 * (norm + px_grad + py_grad) + 4 * 512
    kept.backward()


def test_backward_of_the_recursion_allocates_no_lattices(gpu_device):
    B, S, T = 4, 60, 300
    g = torch.Generator().manual_seed(1)
    px = torch.randn(B, S, T + 1, generator=g).to(gpu_device).requires_grad_(True)
    py = torch.randn(B, S + 1, T, generator=g).to(gpu_device).requires_grad_(True)
    scores, occupation = fast_rnnt_amd.mutual_information_recursion(px, py, return_grad=True)
    total = scores.sum()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    grads = torch.autograd.grad(total, (px, py))
    assert torch.cuda.max_memory_allocated() - before < occupation[0].numel() * 4
    assert all(torch.equal(a, b) for a, b in zip(grads, occupation))


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("B,S,T", [(4, 60, 300), (4, 200, 900)])
def test_memory_that_the_recursion_keeps(gpu_device, B, S, T, modified):
    """One lattice -- not the gradients, which are formed in the backward."""
    g = torch.Generator().manual_seed(2)
    px = torch.randn(B, S, T if modified else T + 1, generator=g).to(gpu_device).requires_grad_(True)
    py = torch.randn(B, S + 1, T, generator=g).to(gpu_device).requires_grad_(True)
    boundary = torch.tensor([[0, 0, S, T]] * B).to(gpu_device)
    fast_rnnt_amd.mutual_information_recursion(px, py, boundary).sum().backward()
    before = torch.cuda.memory_allocated()
    scores = fast_rnnt_amd.mutual_information_recursion(px, py, boundary)
    # (the scores; the shares, with a row for each seam between bands of 64 rows and the boundary's; in multiples of
    # 512 bytes)
    assert torch.cuda.memory_allocated() - before <= 4 * B * (S + 1 + S // 64) * (T + 1) + 32 * B + 2 * 512
    scores.sum().backward()
