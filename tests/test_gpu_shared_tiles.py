"""The normalizer product where two workgroups share a tile, which the losses do on small batches of large
vocabularies, against the entry point that has no workspace for it: the same bits."""
import pytest
import torch

import fast_rnnt_amd as F
from fast_rnnt_amd import _lib

pytestmark = pytest.mark.gpu


def _inputs(B, S, T, C, seed):
    g = torch.Generator().manual_seed(seed)
    am, lm = 3 * torch.randn(B, T, C, generator=g), 3 * torch.randn(B, S + 1, C, generator=g)
    am[0, :, C // 2:] += 40 * torch.rand(C - C // 2, generator=g).cumsum(0)  # (shifts that are raised on the way)
    t_end = (T * (0.5 + 0.5 * torch.rand(B, generator=g))).long().clamp(min=1)
    s_end = torch.minimum((S * (0.5 + 0.5 * torch.rand(B, generator=g))).long().clamp(min=1), t_end)
    zero = torch.zeros_like(t_end)
    boundary = torch.stack([zero, zero, s_end, t_end], 1)
    return am.cuda(), lm.cuda(), torch.randint(0, C, (B, S), generator=g).cuda(), boundary.cuda()


def _without_workspace(lm, am, sym, boundary):
    (B, S1, C), T = lm.shape, am.shape[1]
    S = S1 - 1
    out = {n: torch.empty(s, device="cuda") for n, s in dict(
        px=(B, S, T + 1), py=(B, S1, T), lm_max=(B, S1), am_max=(B, T), norm=(B, S1, T), p=(B, S1, T + 1),
        scores=(B,), gx=(B, S, T + 1), gy=(B, S1, T), loss=(B,)).items()}
    _lib.call("frnnt_simple_loss_fwd_f32", lm.data_ptr(), am.data_ptr(), sym.data_ptr(), _lib.ptr(boundary),
              *(x.data_ptr() for x in out.values()), B, S, T, C, 0, 0, 0, 0, None, _lib.stream_of(am))
    return out["loss"], out["gx"], out["gy"]


# vocabularies of 7 rounds of shares and one entry less (which are not shared), a last slab of one entry and of
# sixteen; one tile, as many as are shared, one more; rows and frames that end at a tile's edge and beside it
@pytest.mark.parametrize("B,S,T,C", [
    (1, 5, 9, 769), (1, 5, 9, 768), (1, 31, 32, 1000), (2, 32, 33, 4097), (1, 63, 64, 5000), (3, 40, 70, 1296),
    (32, 31, 128, 800), (32, 31, 129, 800), (4, 100, 150, 2000), (64, 20, 40, 900)])
def test_shared_tiles_hold_the_same_bits(B, S, T, C):
    am, lm, sym, boundary = _inputs(B, S, T, C, B + S + C)
    for bnd in (boundary, None):
        want = _without_workspace(lm, am, sym, bnd)
        for _ in range(3):  # (a workspace that holds anything, and what the call before has left)
            loss, (gx, gy) = F.rnnt_loss_simple(lm, am, sym, 0, boundary=bnd, reduction="none", return_grad=True)
            for got, expected in zip((loss, gx, gy), want):
                assert torch.equal(got, expected)


def test_shared_tiles_in_a_graph_and_on_two_streams():
    am, lm, sym, boundary = _inputs(3, 40, 100, 2000, 4)
    kinds = dict(boundary=boundary, reduction="none", return_grad=True)
    for x in (am, lm):
        x.requires_grad_(False)
    F.rnnt_loss_simple(lm, am, sym, 0, **kinds)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = F.rnnt_loss_simple(lm, am, sym, 0, **kinds)
    for step in range(4):
        with torch.no_grad():
            lm.mul_(0.9).add_(0.05 * step)
        want_loss, want = F.rnnt_loss_simple(lm, am, sym, 0, **kinds)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded[0], want_loss)
        assert torch.equal(recorded[1][0], want[0]) and torch.equal(recorded[1][1], want[1])
    streams, results = [torch.cuda.Stream() for _ in range(2)], []
    torch.cuda.synchronize()
    for i in range(12):
        with torch.cuda.stream(streams[i % 2]):
            results.append(F.rnnt_loss_simple(lm, am, sym, 0, **kinds))
    torch.cuda.synchronize()
    for loss, (gx, gy) in results:
        assert torch.equal(loss, want_loss) and torch.equal(gx, want[0]) and torch.equal(gy, want[1])


@pytest.mark.parametrize("kind", ["bf16", "lm_only", "modified"])
def test_shared_tiles_of_the_other_losses(kind):
    """The same utterances in a batch too large for shared tiles: the same bits."""
    am, lm, sym, boundary = _inputs(3, 20, 90, 1500, 9)

    def run(copies):
        a, l, y, bnd = (x.repeat(copies, *[1] * (x.dim() - 1)) for x in (am, lm, sym, boundary))
        options = dict(boundary=bnd, reduction="none", return_grad=True)
        if kind == "lm_only":  # (the am-only model has a mean over the batch)
            loss, grads = F.rnnt_loss_smoothed(l, a, y, 0, lm_only_scale=0.25, am_only_scale=0.0, **options)
        elif kind == "bf16":
            loss, grads = F.rnnt_loss_simple(l.bfloat16(), a.bfloat16(), y, 0, **options)
        else:
            loss, grads = F.rnnt_loss_simple(l, a, y, 0, rnnt_type="modified", **options)
        return [x[-3:] for x in (loss, *grads)]

    for got, want in zip(run(1), run(50)):
        assert torch.equal(got, want)


def test_shared_tiles_of_the_smoothed_loss():
    """Both models beside the joint one, against their log-probabilities formed by a call of their own (which
    shares no tile) and the recursion.  A score is a sum over S + T steps of values that round a few times each."""
    am, lm, sym, boundary = _inputs(3, 20, 90, 1500, 11)
    scales = dict(lm_only_scale=0.25, am_only_scale=0.1)
    loss = F.rnnt_loss_smoothed(lm, am, sym, 0, boundary=boundary, reduction="none", **scales)
    px, py = F.get_rnnt_logprobs_smoothed(lm, am, sym, 0, boundary=boundary, **scales)
    want = -F.mutual_information_recursion(px, py, boundary)
    assert bool(((loss - want).abs() <= 8 * (20 + 90) * 2.0 ** -24 * want.abs()).all())
