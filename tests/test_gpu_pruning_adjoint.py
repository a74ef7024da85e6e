"""do_rnnt_pruning's backward where its walk over the frames can go wrong: 1 ... 8 (and more) kept
positions, fewer frames than waves, bounds that jump, stand still, move back or point outside the
lattice, odd and even vocabularies in every type, one gradient for both outputs or two, and the
frames' window starts at the edges of their tiles.  Oracle: indexing and sums in float64."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu
ULP = {torch.float32: 1e-6, torch.float64: 1e-13, torch.float16: 2.0 ** -10,
       torch.bfloat16: 2.0 ** -7}


def _bounds(kind, B, T, S, R, g):
    most = S + 1 - R
    if kind == "anything":
        return torch.randint(-1, S + 2, (B, T, R), generator=g)
    steps = torch.randint(0, {"walk": 2, "jump": 3 * R}[kind], (B, T), generator=g)
    if kind == "jump":
        steps = steps * (torch.rand(B, T, generator=g) < 0.2)
    begin = torch.clamp(torch.cumsum(steps, 1) - steps[:, :1], max=most)
    if B > 1:
        begin[1] = begin[1].flip(0)  # moves back
    return begin.unsqueeze(2) + torch.arange(R)


@pytest.mark.parametrize("dtype", list(ULP))
@pytest.mark.parametrize("B,T,S,R,C", [(1, 1, 1, 1, 1), (2, 7, 5, 2, 63), (3, 40, 30, 3, 130),
                                       (9, 33, 20, 4, 64), (2, 100, 60, 5, 257), (2, 65, 90, 6, 30),
                                       (1, 50, 12, 7, 66), (2, 130, 250, 8, 129), (2, 20, 30, 11, 34)])
def test_pruning_backward(gpu_device, dtype, B, T, S, R, C):
    g = torch.Generator().manual_seed(B * T + S)
    for kind in ("walk", "jump", "anything"):
        ranges = _bounds(kind, B, T, S, R, g)
        am, lm = torch.randn(B, T, C, generator=g), torch.randn(B, S + 1, C, generator=g)
        up = [torch.randn(B, T, R, C, generator=g).to(dtype) for _ in range(2)]
        inside = (ranges >= 0) & (ranges <= S)
        for ga, gl in [(up[0], up[0]), (up[0], up[1]), (None, up[0])]:
            print(f"{dtype} B={B} T={T} S={S} R={R} C={C} {kind}", flush=True)
            a = am.to(dtype).to(gpu_device).requires_grad_(True)
            l = lm.to(dtype).to(gpu_device).requires_grad_(True)
            ap, lp = fast_rnnt_amd.do_rnnt_pruning(a, l, ranges.to(gpu_device))
            assert ap.data_ptr() == a.data_ptr() and ap.shape == lp.shape == (B, T, R, C)
            dev = {id(x): x.to(gpu_device) for x in up}
            outs = [(o, dev[id(x)]) for o, x in ((ap, ga), (lp, gl)) if x is not None]
            torch.autograd.backward([o for o, _ in outs], [x for _, x in outs])
            rows = torch.where(inside, ranges, torch.full_like(ranges, S + 1))
            want = torch.zeros(B, S + 2, C, dtype=torch.float64)
            want.scatter_add_(1, rows.reshape(B, T * R, 1).expand(B, T * R, C),
                              gl.double().reshape(B, T * R, C))
            size = torch.zeros(B, S + 2, C, dtype=torch.float64)
            size.scatter_add_(1, rows.reshape(B, T * R, 1).expand(B, T * R, C),
                              gl.double().abs().reshape(B, T * R, C))
            off = (l.grad.double().cpu() - want[:, :S + 1]).abs()
            assert bool((off <= ULP[dtype] * size[:, :S + 1] + 1e-30).all())
            if ga is not None:
                off = (a.grad.double().cpu() - ga.double().sum(2)).abs()
                assert bool((off <= ULP[dtype] * ga.double().abs().sum(2)).all())
            else:
                assert a.grad is None


@pytest.mark.parametrize("T", [31, 32, 33, 64, 97])
@pytest.mark.parametrize("S", [1, 7, 8, 63, 64, 120])
def test_window_starts_at_the_edges_of_tiles(gpu_device, T, S):
    g = torch.Generator().manual_seed(T + S)
    B = 2
    gx, gy = torch.rand(B, S, T + 1, generator=g), torch.rand(B, S + 1, T, generator=g)
    boundary = torch.tensor([[0, 0, S, T], [0, 0, max(1, S - 2), T - 1]])
    for R in (2, min(5, S + 1)):
        print(f"T={T} S={S} R={R}", flush=True)
        got = fast_rnnt_amd.get_rnnt_prune_ranges(gx.to(gpu_device), gy.to(gpu_device),
                                                  boundary.to(gpu_device), R).cpu()
        assert torch.equal(got, O.prune_ranges(gx, gy, boundary, R))
