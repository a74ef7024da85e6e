"""The kernels that take several short logits rows per wave, forward and backward, which large batches run, against
those with a row per wave, which the same utterances run in a small batch: the same bits.  Row lengths at the edges of
a quarter, a half and a whole wave of 16-byte pieces, rows that begin anywhere in a piece, windows, ranges, rows of
infinities and NaN, and frame counts that end inside a wave's rows."""
import pytest
import torch

import fast_rnnt_amd as F

pytestmark = pytest.mark.gpu


def _case(B, T, S, R, C, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    sym = torch.randint(0, C, (B, S), generator=g)
    t_end = torch.tensor([T, max(1, T - 5), max(1, T // 2)])[:B]
    s_end = torch.minimum(torch.tensor([S, max(1, S - 2), max(1, S // 2)])[:B], t_end)
    zero = torch.zeros_like(t_end)
    logits = 3 * torch.randn(B, T, R, C, generator=g)
    logits[0, T // 3, R // 2, C // 2] = float("inf")
    logits[0, T // 4, 0, 0] = float("nan")
    logits[1, T // 5, R - 1] = -float("inf")
    return logits.to(dtype).cuda(), sym.cuda(), torch.stack([zero, zero, s_end, t_end], 1).cuda()


# (the last copy begins where the first does within a 16-byte piece, eight copies being a multiple of 16 bytes: what
# a lane sums depends on it)
def _run(fn, logits, copies, offset, *args, **kwargs):
    x = logits.repeat(copies, 1, 1, 1)
    memory = torch.empty(x.numel() + offset, dtype=x.dtype, device="cuda")
    x = memory[offset:].view(x.shape).copy_(x).requires_grad_()
    args = [a.repeat(copies, *[1] * (a.dim() - 1)) for a in args]
    boundary = args.pop()
    loss = fn(x, *args, 0, boundary=boundary, reduction="none", **kwargs)
    weights = torch.linspace(0.5, 2, logits.shape[0], device="cuda").repeat(copies)
    (grad,) = torch.autograd.grad((weights * loss).sum(), x)
    n = logits.shape[0]
    return [y[k * n:(k + 1) * n] for k in (0, copies - 1) for y in (loss.detach(), grad)]


def _same(a, b):
    return torch.equal(torch.nan_to_num(a, nan=12345.0), torch.nan_to_num(b, nan=12345.0))


@pytest.mark.parametrize("dtype,lengths", [
    (torch.float32, (1, 60, 61, 64, 65, 113, 128, 129, 200, 255, 256, 257, 333, 500, 512, 513, 750, 768)),
    (torch.float16, (9, 121, 128, 130, 250, 256, 302, 504, 512)),
    (torch.bfloat16, (8, 80, 127, 136, 249, 255, 303, 505, 511))])
@pytest.mark.parametrize("offset", [0, 3])
def test_pruned_rows_hold_the_same_bits(dtype, lengths, offset):
    B, T, S, R = 3, 37, 12, 5
    for C in lengths:
        logits, sym, boundary = _case(B, T, S, R, C, dtype, C)
        begin = torch.linspace(0, S + 1 - R, T, device="cuda").long().expand(B, T)
        ranges = begin.unsqueeze(2) + torch.arange(R, device="cuda")
        for kind in ("regular", "constrained"):
            few = _run(F.rnnt_loss_pruned, logits, 1, offset, sym, ranges, boundary, rnnt_type=kind)
            many = _run(F.rnnt_loss_pruned, logits, 153, offset, sym, ranges, boundary, rnnt_type=kind)
            assert all(_same(a, b) for a, b in zip(few, many))


@pytest.mark.parametrize("dtype,C", [(torch.float32, 64), (torch.float32, 101), (torch.float32, 300),
                                     (torch.bfloat16, 238)])
def test_rows_of_the_whole_lattice_hold_the_same_bits(dtype, C):
    logits, sym, boundary = _case(2, 31, 10, 11, C, dtype, C)
    few = _run(F.rnnt_loss, logits, 1, 0, sym, boundary)
    many = _run(F.rnnt_loss, logits, 153, 0, sym, boundary)
    assert all(_same(a, b) for a, b in zip(few, many))
