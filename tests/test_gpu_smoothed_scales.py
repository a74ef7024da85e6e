"""rnnt_loss_smoothed's row statistics and interpolation, which are formed before and within the
normalizer product: vocabularies around the 512 entries that a wave holds in registers, batches of rows
around its blocks of 16, no am-only model against one of no weight, and what is not finite."""
import math

import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu


def _case(B, S, T, C, seed=0):
    g = torch.Generator().manual_seed(seed + B + S + T + C)
    lm, am = 2 * torch.randn(B, S + 1, C, generator=g), 2 * torch.randn(B, T, C, generator=g)
    symbols = torch.randint(1, C, (B, S), generator=g)
    t_end = torch.tensor([T] + [max(S, T - 3 * b) for b in range(1, B)])
    s_end = torch.tensor([S] + [max(1, S - b) for b in range(1, B)])
    zero = torch.zeros(B, dtype=torch.long)
    return lm, am, symbols, torch.stack([zero, zero, s_end, t_end], 1)


def _run(f, lm, am, symbols, boundary, dev=None, **args):
    x = [(v.to(dev) if dev else v.clone()).requires_grad_(True) for v in (lm, am)]
    to = (lambda v: v.to(dev)) if dev else (lambda v: v)
    loss = f(*x, to(symbols), 0, boundary=to(boundary), reduction="none", **args)
    loss.sum().backward()
    return [v.detach().cpu() for v in (loss, x[0].grad, x[1].grad)]


@pytest.mark.parametrize("am_scale", [0.0, 0.15])
@pytest.mark.parametrize("B,S,T,C", [(1, 15, 20, 511), (2, 7, 33, 512), (3, 10, 31, 513), (2, 31, 70, 1030)])
def test_statistics_of_rows_in_and_out_of_registers(gpu_device, B, S, T, C, am_scale):
    case = _case(B, S, T, C)
    args = dict(lm_only_scale=0.25, am_only_scale=am_scale, delay_penalty=0.01)
    want = _run(O.loss_smoothed, *case, **args)
    got = _run(fast_rnnt_amd.rnnt_loss_smoothed, *case, dev=gpu_device, **args)
    # scores of some hundred nats in float32: occupations to 2e-5 of them (as in the tests beside this)
    assert torch.allclose(got[0], want[0], rtol=1e-5, atol=1e-5)
    for x, y in zip(got[1:], want[1:]):
        assert bool(((x - y).abs() <= 2e-4 + 1e-4 * y.abs()).all()), (x - y).abs().max().item()


@pytest.mark.parametrize("kind", ["regular", "modified"])
def test_no_am_model_is_one_of_no_weight(gpu_device, kind):
    # 0 (no model is formed) against 1e-18 (formed, and below a unit in the last place of all it is added to)
    case = _case(3, 40, 90, 200)
    args = dict(lm_only_scale=0.25, rnnt_type=kind, delay_penalty=0.01)
    none, weightless = [_run(fast_rnnt_amd.rnnt_loss_smoothed, *case, dev=gpu_device, am_only_scale=a,
                             **args) for a in (0.0, 1e-18)]
    assert torch.equal(none[0], weightless[0])
    # the gradients get terms of 1e-18 from the second, below half a unit of anything above 1e-10
    for x, y in zip(none[1:], weightless[1:]):
        assert bool(((x - y).abs() <= 1e-15 + 2.0 ** -23 * y.abs()).all())


@pytest.mark.parametrize("am_scale", [0.0, 0.15])
def test_one_bad_row_of_lm_reaches_every_utterance(gpu_device, am_scale):
    # through the unigram, a mean over all rows of the batch, padding rows included (rnnt_loss.py:1278-1281)
    lm, am, symbols, boundary = _case(3, 20, 40, 60)
    for value in (math.nan, math.inf):
        bad = lm.clone()
        bad[2, 20, 5] = value  # (a row of padding)
        args = dict(lm_only_scale=0.25, am_only_scale=am_scale)
        want = _run(O.loss_smoothed, bad, am, symbols, boundary, **args)
        got = _run(fast_rnnt_amd.rnnt_loss_smoothed, bad, am, symbols, boundary, dev=gpu_device, **args)
        # (the recursion's log-add takes the larger operand past a NaN: infinite here, a NaN there)
        assert not bool(want[0].isfinite().any()) and not bool(got[0].isfinite().any())
        assert bool(got[1].isnan().all())
        for b in range(3):  # (frames past the window get exact zeros)
            end = int(boundary[b, 3])
            assert bool(got[2][b, :end].isnan().all()) and not bool(got[2][b, end:].any())


@pytest.mark.parametrize("am_scale", [0.0, 0.15])
def test_entries_of_minus_infinity(gpu_device, am_scale):
    # a symbol that a frame rules out: px is -inf there, as in the reference, with either scale
    lm, am, symbols, boundary = _case(2, 9, 30, 40)
    am[:, 3, :] = am[:, 3, :].masked_fill(torch.arange(40) > 20, -math.inf)
    args = dict(lm_only_scale=0.25, am_only_scale=am_scale)
    want = _run(O.loss_smoothed, lm, am, symbols, boundary, **args)
    got = _run(fast_rnnt_amd.rnnt_loss_smoothed, lm, am, symbols, boundary, dev=gpu_device, **args)
    assert torch.allclose(got[0], want[0], rtol=1e-5, atol=1e-5)
    for x, y in zip(got[1:], want[1:]):
        fine = y.isfinite()
        assert bool(((x - y).abs() <= 2e-4 + 1e-4 * y.abs())[fine].all())
