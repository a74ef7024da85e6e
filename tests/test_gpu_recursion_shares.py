"""The recursion of the losses, which leaves the shares of the cells' gradients in the place of p, against
the two entry points that go through p: the same operations, so the same bits."""
import math

import pytest
import torch

import fast_rnnt_amd as F
from fast_rnnt_amd import _fast_rnnt, _lib

pytestmark = pytest.mark.gpu


def _inputs(B, S, T, modified, seed):
    g = torch.Generator().manual_seed(seed)
    T1 = T if modified else T + 1
    px = -2.0 + 1.5 * torch.randn(B, S, T1, generator=g)
    py = -1.0 + torch.randn(B, S + 1, T, generator=g)
    if not modified:
        px[:, :, T] = -math.inf
    return px, py, g


def _window(B, S, T, g):
    rows = []
    for _ in range(B):
        s0 = int(torch.randint(0, S // 3 + 1, (), generator=g))
        t0 = int(torch.randint(0, T // 3 + 1, (), generator=g))
        rows.append([s0, t0, int(torch.randint(s0, S + 1, (), generator=g)),
                     int(torch.randint(t0, T + 1, (), generator=g))])
    rows[0] = [0, 0, S, T]
    return torch.tensor(rows)


def _pair(px, py, boundary, held, kept):
    """Scores and gradients of ones from the kernels that pass shares, whatever a loss of this size takes; the buffer
    between them is full of `held`, and so are the gradients'."""
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    B, S, T = px.shape[0], px.shape[1], py.shape[2]
    sizes = B, S, T, int(px.shape[2] == T)
    n = lib.frnnt_mi_kept_size(B, S, T) if kept else B * (S + 1) * (T + 1)
    shares, scores = torch.full((n,), held, device="cuda"), torch.full((B,), held, device="cuda")
    gx, gy = torch.full_like(px, held), torch.full_like(py, held)
    ins = px.data_ptr(), py.data_ptr(), None if boundary is None else boundary.data_ptr()
    if kept:
        assert lib.frnnt_mi_kept_fwd_f32(*ins, shares.data_ptr(), scores.data_ptr(), *sizes, 0, None, stream) == 0
        assert lib.frnnt_mi_kept_bwd_f32(shares.data_ptr(), int(boundary is not None), None, 0, gx.data_ptr(),
                                         gy.data_ptr(), *sizes, stream) == 0
    else:
        assert lib.frnnt_mi_shares_fwd_f32(*ins, shares.data_ptr(), scores.data_ptr(), None, gy.data_ptr(), *sizes, 0,
                                           None, stream) == 0
        assert lib.frnnt_mi_shares_bwd_f32(ins[2], shares.data_ptr(), None, 0, gx.data_ptr(), gy.data_ptr(), *sizes,
                                           stream) == 0
    return scores, gx, gy


def _compare(px, py, boundary, held=math.nan):
    """The pair in both its forms, and whichever kernels a loss of this size takes, against the two through p."""
    px, py = px.cuda(), py.cuda()
    boundary = None if boundary is None else boundary.cuda()
    B, S, T = px.shape[0], px.shape[1], py.shape[2]
    p = torch.empty(B, S + 1, T + 1, device="cuda")
    want = _fast_rnnt.mutual_information_forward(px, py, boundary, p)
    want_x, want_y = _fast_rnnt.mutual_information_backward(px, py, boundary, p,
                                                            torch.ones(B, device="cuda"))
    score, grads = F.mutual_information_recursion(px, py, boundary, return_grad=True)
    for got in ((score, *grads), _pair(px, py, boundary, held, False), _pair(px, py, boundary, held, True)):
        for a, b in zip(got, (want, want_x, want_y)):
            assert torch.allclose(a, b, rtol=0, atol=0, equal_nan=True)
    return want_x, want_y


# one step to a tile's remainder either way, one row to a band's, one to four bands in a workgroup or
# apart, more than four
@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("B,S,T", [
    (2, 1, 1), (5, 7, 31), (4, 30, 33), (3, 62, 64), (3, 63, 65), (3, 64, 95), (2, 65, 160),
    (9, 127, 130), (2, 128, 191), (2, 200, 257), (3, 255, 1100), (2, 300, 310), (130, 66, 300), (2, 70, 900),
    (4, 100, 770), (3, 200, 100),
])
def test_same_bits_as_through_p(B, S, T, modified):
    px, py, g = _inputs(B, S, T, modified, 17 * S + T)
    _compare(px, py, None)
    _compare(px, py, _window(B, S, T, g))


# cells whose share is not finite pass nothing on; cells that cannot be reached hand everything left
@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T", [(20, 40), (63, 150), (64, 150), (150, 200), (130, 1300)])
@pytest.mark.parametrize("value", [math.nan, math.inf, -math.inf])
def test_cells_that_are_not_finite(S, T, modified, value):
    px, py, g = _inputs(6, S, T, modified, S + T)
    for b in range(1, 6):  # 1, 4, 16, ... cells of px, or of px and py; utterance 0 stays as it is
        for x in (px, py)[:1 + b % 2]:
            flat = x[b].reshape(-1)
            flat[torch.randint(0, flat.numel(), (4 ** (b - 1),), generator=g)] = value
    _compare(px, py, None)
    _compare(px, py, _window(6, S, T, g))


@pytest.mark.parametrize("modified", [False, True])
def test_lattice_without_a_path(modified):
    px, py, _ = _inputs(3, 90, 120, modified, 3)
    px[1, 40] = -math.inf  # no way from row 40 to row 41
    py[2] = -math.inf
    px[2] = -math.inf
    _compare(px, py, None)


# memory that the scratch is made of may hold anything: cells around the windows must not be felt
@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T", [(40, 90), (100, 140), (150, 300), (100, 1300), (300, 310)])
@pytest.mark.parametrize("value", [math.nan, math.inf, -3.0, 3e38])
def test_what_the_scratch_held_before(S, T, modified, value):
    px, py, g = _inputs(8, S, T, modified, 9)
    boundary = _window(8, S, T, g)
    want_x, want_y = _compare(px, py, boundary, value)
    assert torch.isfinite(want_x).all() and torch.isfinite(want_y).all()


# one band, two together, two, three and four apart, two apart in the backward alone, four in the forward alone
@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("B,S,T", [(5, 20, 33), (5, 100, 90), (4, 100, 1300), (4, 150, 200), (3, 250, 700),
                                   (4, 100, 770), (3, 200, 100)])
def test_backward_again_on_the_same_shares(B, S, T, modified, kept):
    """With another gradient of the scores, into buffers that hold anything, those of the first call among them: what
    a first call on shares of their own forms.  With and without the room behind the shares."""
    px, py, g = _inputs(B, S, T, modified, S)
    px, py, boundary = px.cuda(), py.cuda(), _window(B, S, T, g).cuda()
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    room = lib.frnnt_mi_kept_size(B, S, T)
    assert room >= B * (S + 1) * (T + 1)

    def forward():
        shares = torch.full((room if kept else B * (S + 1) * (T + 1),), 7.0, device="cuda")
        scores, scratch = torch.empty(B, device="cuda"), torch.empty_like(py)
        ins, rest = [x.data_ptr() for x in (px, py, boundary, shares, scores)], (B, S, T, int(modified), 0, None, stream)
        rc = (lib.frnnt_mi_kept_fwd_f32(*ins, *rest) if kept else
              lib.frnnt_mi_shares_fwd_f32(*ins, None, scratch.data_ptr(), *rest))
        assert rc == 0
        return shares

    def backward(shares, seeds, grads):
        rest = (seeds.data_ptr(), 1, grads[0].data_ptr(), grads[1].data_ptr(), B, S, T, int(modified), stream)
        rc = (lib.frnnt_mi_kept_bwd_f32(shares.data_ptr(), 1, *rest) if kept else
              lib.frnnt_mi_shares_bwd_f32(boundary.data_ptr(), shares.data_ptr(), *rest))
        assert rc == 0
        return [x.clone() for x in grads]

    one, two = torch.linspace(1, 3, B, device="cuda"), torch.linspace(-2, 0.5, B, device="cuda")
    shares, grads = forward(), [torch.full_like(px, 7.0), torch.full_like(py, 7.0)]
    first, second, third = (backward(shares, seeds, grads) for seeds in (one, two, one))
    want = backward(forward(), two, [torch.zeros_like(px), torch.zeros_like(py)])
    occ = F.mutual_information_recursion(px, py, boundary, return_grad=True)[1]
    for a, b, c, w, o in zip(first, second, third, want, occ):
        assert torch.equal(a, c) and torch.equal(b, w)
        assert torch.allclose(b, o * two.reshape(-1, 1, 1), rtol=2 * (S + T) * 2.0 ** -24, atol=1e-37)


@pytest.mark.parametrize("B,S,T", [(6, 40, 150), (6, 80, 250), (8, 100, 900), (8, 250, 700)])
def test_a_wait_that_runs_out_shows_as_nan(B, S, T):
    """With the bound of the kernels' waits set from the host: an utterance's score is NaN, or its gradients
    hold one, unless everything is what it is without a bound."""
    px, py, _ = _inputs(B, S, T, False, S)
    px, py = px.cuda(), py.cuda()
    score, (gx, gy) = F.mutual_information_recursion(px, py, None, return_grad=True)
    lib = _lib.load()
    gave_up = 0
    for polls in (1, 3, 10, 40, 150, 600, 1 << 22):
        lib.frnnt_set_spin_limit(polls)
        try:
            score1, (gx1, gy1) = F.mutual_information_recursion(px, py, None, return_grad=True)
            torch.cuda.synchronize()
        finally:
            lib.frnnt_set_spin_limit(0)
        for b in range(B):
            failed = bool(torch.isnan(score1[b]))
            gave_up += failed
            if failed:
                continue
            assert torch.equal(score1[b], score[b])
            nan = bool(torch.isnan(gx1[b]).any()), bool(torch.isnan(gy1[b]).any())
            assert all(nan) or (torch.equal(gx1[b], gx[b]) and torch.equal(gy1[b], gy[b]))
        assert polls > 1 or gave_up == B
        assert polls < 1 << 22 or (torch.equal(score1, score) and torch.equal(gx1, gx))


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("B,S,T", [(4, 9, 20), (5, 70, 100), (4, 130, 1200)])
def test_gradients_formed_in_the_backward(B, S, T, modified):
    """Without return_grad the occupation gradients are formed in the backward, from the gradient of the
    scores: against those that are formed in the forward and scaled.  A factor that is a power of two
    commutes with every rounding but those of subnormal numbers, by 2^-149 per step of a path; another
    one rounds once per step at most, S + T of them."""
    px, py, g = _inputs(B, S, T, modified, S)
    px, py, boundary = px.cuda(), py.cuda(), _window(B, S, T, g).cuda()
    powers = torch.tensor([-1.0, 0.25, 2.0, 0.0, -4.0])[:B].cuda()
    anything = torch.randn(B, generator=g).cuda()

    def grads(factor, return_grad):
        x, y = px.clone().requires_grad_(), py.clone().requires_grad_()
        out = F.mutual_information_recursion(x, y, boundary, return_grad=return_grad)
        (out[0] if return_grad else out).backward(factor)
        return x.grad, y.grad

    for factor in (powers, anything, powers[1:2].expand(B)):
        want, got = grads(factor, True), grads(factor, False)
        for w, h in zip(want, got):
            if factor is anything:
                assert torch.allclose(h, w, rtol=2 * (S + T) * 2.0 ** -24, atol=1e-37)
            else:
                assert torch.allclose(h, w, rtol=0, atol=4 * (S + T) * 2.0 ** -149)
    for value in (float("nan"), float("inf")):
        factor = anything.clone()
        factor[1] = value
        for w, h in zip(grads(factor, True), grads(factor, False)):
            assert not torch.isfinite(h[1]).any() and not torch.isfinite(w[1]).any()
            assert torch.isfinite(h[0]).all()

    x, y = px.clone().requires_grad_(), py.clone().requires_grad_()
    total = -F.mutual_information_recursion(x, y, boundary).sum()
    total.backward(retain_graph=True)
    with pytest.raises(RuntimeError):  # scaled in place, as after the reference's "*="
        total.backward()


def test_gradient_of_a_gradient_formed_in_the_backward():
    px, py, _ = _inputs(3, 12, 30, False, 5)
    px, py = px.cuda(), py.cuda()
    _, (occ_x, _) = F.mutual_information_recursion(px, py, None, return_grad=True)
    x, y = px.clone().requires_grad_(), py.clone().requires_grad_()
    weight = torch.tensor([0.5, 1.0, 2.0], device="cuda", requires_grad=True)
    loss = (weight * F.mutual_information_recursion(x, y)).sum()
    (gx,) = torch.autograd.grad(loss, x, create_graph=True)
    assert torch.equal(gx.detach(), occ_x * weight.detach().reshape(-1, 1, 1))
    (gw,) = torch.autograd.grad(gx.sum(), weight)
    assert torch.allclose(gw, occ_x.sum(dim=(1, 2)), rtol=1e-5)


@pytest.mark.parametrize("B,S,T", [(5, 100, 90), (4, 150, 300)])
def test_recursion_and_its_backward_in_a_graph(B, S, T):
    """Replays on other inputs, with eager calls between them: each finds the room between the workgroups as it
    was."""
    px, py, g = _inputs(B, S, T, False, S)
    px, py, boundary = px.cuda(), py.cuda(), _window(B, S, T, g).cuda()
    seeds = torch.linspace(0.5, 2, B, device="cuda")

    def step():
        x, y = px.detach().requires_grad_(), py.detach().requires_grad_()
        scores = F.mutual_information_recursion(x, y, boundary)
        return scores.detach(), *torch.autograd.grad(scores, (x, y), seeds)

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(3):
        px.add_(0.25)
        want = step()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("B,S,T", [(1, 1, 1), (5, 20, 33), (5, 100, 90), (4, 150, 300), (3, 300, 320)])
def test_boundary_written_to_between_forward_and_backward(B, S, T, modified):
    """A program may fill one boundary buffer for one recursion after the other, as when the gradients were formed in
    the forward: they are those of the rows that the scores were formed with."""
    px, py, g = _inputs(B, S, T, modified, S)
    px, py = px.cuda().requires_grad_(), py.cuda().requires_grad_()
    one, two = _window(B, S, T, g).cuda(), _window(B, S, T, g).flip(0).cuda()
    want = [torch.autograd.grad(F.mutual_information_recursion(px, py, rows.clone()).sum(), (px, py))
            for rows in (one, two)]
    buffer = one.clone()
    first = F.mutual_information_recursion(px, py, buffer)
    buffer.copy_(two)
    second = F.mutual_information_recursion(px, py, buffer)
    buffer.zero_()
    for scores, grads in ((second, want[1]), (first, want[0])):
        for a, b in zip(torch.autograd.grad(scores.sum(), (px, py)), grads):
            assert torch.equal(a, b)
