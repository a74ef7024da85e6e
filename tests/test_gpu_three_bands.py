"""Three bands of 64 rows in workgroups of their own on lattices of any length, which small batches of the recursion and
of the losses that pass shares run, against one workgroup per utterance, which the same utterances run in a batch too
large for that: the same bits.  Windows that leave bands out, are empty or start inside the lattice; one frame."""
import pytest
import torch

import fast_rnnt_amd as F
from fast_rnnt_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T", [(128, 1), (128, 31), (129, 64), (150, 33), (130, 140), (160, 160), (191, 200), (191, 300)])
def test_three_bands_of_any_length(gpu_device, S, T, modified):
    g = torch.Generator().manual_seed(S + T)
    rows = [[0, 0, S, T], [0, 0, S, max(1, T - 1)], [0, 0, 63, T], [0, 0, 64, T], [0, 0, 127, T], [0, 0, 128, T],
            [2, T // 3, S - 1, T], [0, 0, S, 0]]
    n, T1 = len(rows), T if modified else T + 1
    px, py = -1 + torch.randn(n, S, T1, generator=g), -1 + torch.randn(n, S + 1, T, generator=g)

    def run(copies, apart):
        # (the recursion always passes shares if its gradients are not handed out; a loss, and what is handed out,
        # from some length on)
        assert _lib.load().frnnt_mi_route(n * copies, S, T, 1) & 3 == apart
        x, y = (v.to(gpu_device).repeat(copies, 1, 1).requires_grad_() for v in (px, py))
        boundary = torch.tensor(rows).to(gpu_device).repeat(copies, 1)
        handed_out, (gx, gy) = F.mutual_information_recursion(x, y, boundary, return_grad=True)
        scores = F.mutual_information_recursion(x, y, boundary)
        seeds = torch.linspace(0.5, 2, n, device=gpu_device).repeat(copies)
        formed = torch.autograd.grad(scores, (x, y), seeds)
        return [v[-n:].cpu() for v in (handed_out.detach(), scores.detach(), gx, gy, *formed,
                                       *torch.autograd.grad(handed_out, (x, y), seeds))]

    for a, b in zip(run(1, 3), run(12, 0)):
        assert torch.equal(torch.nan_to_num(a, nan=1e30), torch.nan_to_num(b, nan=1e30))


def test_three_bands_in_a_graph_and_in_a_loss(gpu_device):
    """Replays find the marks of their own launch; the loss of a batch is formed beside the bands."""
    B, S, T, C = 4, 140, 150, 20
    g = torch.Generator().manual_seed(3)
    lm, am = (torch.randn(B, n, C, generator=g).to(gpu_device) for n in (S + 1, T))
    sym = torch.randint(0, C, (B, S), generator=g).to(gpu_device)
    many = [x.repeat(25, 1, 1) for x in (lm, am)]
    want, grads = F.rnnt_loss_simple(*many, sym.repeat(25, 1), 0, reduction="none", return_grad=True)
    graph = torch.cuda.CUDAGraph()
    F.rnnt_loss_simple(lm, am, sym, 0, reduction="none", return_grad=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        loss, (gx, gy) = F.rnnt_loss_simple(lm, am, sym, 0, reduction="none", return_grad=True)
    for _ in range(3):
        gx.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(loss, want[:B]) and torch.equal(gx, grads[0][:B]) and torch.equal(gy, grads[1][:B])
