"""Which launch the recursion takes, at both sides of the lines that the comments beside the rules give figures for
(host only)."""
import pytest

from fast_rnnt_amd import _lib

FORWARD, BACKWARD, LOSS_SHARES = 1, 2, 4


def _route(B, S, T, shares):
    return _lib.load().frnnt_mi_route(B, S, T, int(shares))


@pytest.mark.parametrize("S,T", [(70, 3000), (100, 1500), (127, 2990), (100, 3100), (127, 12000)])
def test_two_bands_that_pass_shares_have_a_compute_unit_each_or_stay_together(S, T):
    """Of the workgroups of that launch only one fits a compute unit, at any length."""
    apart = FORWARD | BACKWARD
    assert _route(128, S, T, True) & apart == apart
    for B in (129, 160, 256, 300):
        assert _route(B, S, T, True) & apart == 0


@pytest.mark.parametrize("S,T,B", [(130, 1500, 100), (190, 3000, 168), (250, 1500, 128)])
def test_more_bands_stay_apart_with_two_to_a_unit(S, T, B):
    assert _route(B, S, T, True) & FORWARD and _route(B, S, T, True) & BACKWARD


@pytest.mark.parametrize("B,S,T,pays", [
    (3, 63, 1, True), (3, 64, 199, False), (3, 127, 200, True), (2, 128, 119, False), (2, 255, 120, True),
    (100, 130, 399, False), (100, 130, 400, True), (2, 256, 399, False), (2, 300, 400, True),
])
def test_where_losses_pass_shares(B, S, T, pays):
    assert bool(_route(B, S, T, True) & LOSS_SHARES) == pays


def test_bad_sizes_are_refused():
    assert _route(0, 1, 1, False) < 0 and _route(1, -1, 1, True) < 0
