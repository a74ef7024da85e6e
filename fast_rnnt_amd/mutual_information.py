"""Autograd front end of the lattice recursion.

Same public functions, arguments, return values and assertion behaviour as
fast_rnnt/python/fast_rnnt/mutual_information.py; the work is done by the
gfx950 operators in :mod:`fast_rnnt_amd._fast_rnnt`.

The recursion, for the window ``[s_begin, t_begin, s_end, t_end]`` of each batch
row (default ``[0, 0, S, T]``)::

    p[b, s_begin, t_begin] = 0
    p[b, s, t] = log_add(p[b, s-1, t] + px[b, s-1, t],      # px has T+1 columns
                         p[b, s, t-1] + py[b, s, t-1])
    p[b, s, t] = log_add(p[b, s-1, t-1] + px[b, s-1, t-1],  # px has T columns ("modified")
                         p[b, s, t-1] + py[b, s, t-1])

with out-of-window terms taken as -inf; the result is ``p[b, s_end, t_end]``.
"""
import weakref
from typing import List, Optional, Sequence, Tuple, Union

import torch
from torch import Tensor

from . import _fast_rnnt, _lib


_rows_cache = []  # [(weakref to the tensor, its version counter, rows, the rows as a host tensor)]


def boundary_rows(boundary: Tensor, reread: bool = False):
    """``boundary.tolist()``, remembered per tensor object and version counter, so that
    the validity checks of one loss call (and of repeated calls with the same boundary
    tensor, e.g. the smoothed and the pruned loss of one training step) copy the rows
    from the device only once.  Every in-place torch operation bumps the version
    counter; a writer that bypasses it (``.data``, a raw-pointer kernel) must pass
    ``reread=True`` once, or call :func:`forget_boundary_rows`."""
    return _boundary_entry(boundary, reread)[2]


def boundary_on_host(boundary: Tensor) -> Tensor:
    """The host copy behind :func:`boundary_rows`, as a tensor."""
    return _boundary_entry(boundary, False)[3]


def _boundary_entry(boundary, reread):
    version = boundary._version
    if not reread:
        for entry in _rows_cache:
            if entry[0]() is boundary and entry[1] == version:
                return entry
    host = boundary.detach().cpu().contiguous()
    _rows_cache[:] = [e for e in _rows_cache if e[0]() is not boundary and e[0]() is not None]
    _rows_cache.insert(0, (weakref.ref(boundary), version, host.tolist(), host))
    del _rows_cache[8:]
    return _rows_cache[0]


def forget_boundary_rows() -> None:
    """Drop every remembered host copy of a boundary tensor."""
    del _rows_cache[:]


def _assert_boundary(boundary: Tensor, B: int, S: int, T: int, on_device: bool = False) -> None:
    """The boundary assertions of mutual_information.py:277-288.  ``on_device``: the rows
    are left to the recursion's forward kernel, which tests every row anyway (a bad one is
    skipped, its score becomes nan) and reports a failure to the host, where it is raised
    as an AssertionError by a later call or by :func:`check_boundaries`."""
    assert boundary.dtype == torch.int64
    assert boundary.shape == (B, 4)
    if on_device:
        return
    for s_begin, t_begin, s_end, t_end in boundary_rows(boundary):
        assert 0 <= s_begin <= s_end <= S
        assert 0 <= t_begin <= t_end <= T


def set_boundary_checks(mode: str) -> None:
    """Where the rows of a ``boundary`` tensor are asserted.

    ``"device"`` (the default): by the recursion's forward kernel.  A call with a bad row
    returns nan for that row's score, and the reference's ``AssertionError`` is raised by
    the next call into this package on that GPU, or by :func:`check_boundaries` -- no call
    waits for the device.  ``"host"``: before the call, from ``boundary.tolist()``, as the
    reference does (mutual_information.py:277-288, rnnt_loss.py:25-42); every call with a
    boundary tensor it has not seen then waits for the device.
    """
    if mode not in ("device", "host"):
        raise ValueError(f"mode should be ('device' | 'host'), given {mode}")
    _lib.ops().set_deferred_checks(mode == "device")


def check_boundaries(device=None) -> None:
    """Wait for the GPU and raise the ``AssertionError`` of a boundary row that one of the
    calls so far has found bad on the device (see :func:`set_boundary_checks`)."""
    index = torch.cuda.current_device() if device is None else torch.device(device).index
    _lib.ops().check_boundaries(int(index))


class MutualInformationRecursionFunction(torch.autograd.Function):
    """The reference's autograd wrapper under its own name
    (fast_rnnt/python/fast_rnnt/mutual_information.py:24-181), for code that calls ``.apply``;
    :func:`mutual_information_recursion` itself goes through a compiled node of the same behaviour.

    ``forward`` runs the forward operator and, when gradients may be needed, immediately the
    backward operator with a gradient of ones, whose results also go into the caller's list
    ``pxy_grads`` of two; ``backward`` only scales them, in place.
    """

    @staticmethod
    def forward(ctx, px: Tensor, py: Tensor, pxy_grads: List[Optional[Tensor]],
                boundary: Optional[Tensor] = None, return_grad: bool = False) -> Tensor:
        (B, S, T1) = px.shape
        T = py.shape[-1]
        assert T1 in [T, T + 1]
        assert py.shape == (B, S + 1, T)
        if boundary is not None:
            assert boundary.shape == (B, 4)
        assert len(pxy_grads) == 2
        p = torch.empty(B, S + 1, T + 1, device=px.device, dtype=px.dtype)
        scores = _fast_rnnt.mutual_information_forward(px, py, boundary, p)
        grads = [None, None]
        if return_grad or px.requires_grad or py.requires_grad:
            grads = _fast_rnnt.mutual_information_backward(px, py, boundary, p,
                                                           torch.ones_like(scores))
            ctx.save_for_backward(*grads)
        pxy_grads[:] = grads
        return scores

    @staticmethod
    def backward(ctx, ans_grad: Tensor) -> Tuple[Tensor, Tensor, None, None, None]:
        px_grad, py_grad = ctx.saved_tensors
        scale = ans_grad.reshape(-1, 1, 1)
        px_grad *= scale
        py_grad *= scale
        return px_grad, py_grad, None, None, None


def mutual_information_recursion(
    px: Tensor, py: Tensor, boundary: Optional[Tensor] = None, return_grad: bool = False,
) -> Union[Tuple[Tensor, Tuple[Tensor, Tensor]], Tensor]:
    """fast_rnnt/python/fast_rnnt/mutual_information.py:184-298.

    Args:
      px: ``[B][S][T+1]`` (or ``[B][S][T]`` for the modified lattice) log-odds of
        extending the x sequence at lattice position (s, t).
      py: ``[B][S+1][T]`` log-odds of extending the y sequence.
      boundary: optional int64 ``[B][4]`` rows ``[s_begin, t_begin, s_end, t_end]``.
      return_grad: also return ``(px_grad, py_grad)``, the occupation
        probabilities, i.e. the gradients of ``scores.sum()``.
    Returns:
      ``scores`` of shape ``[B]``, or ``(scores, (px_grad, py_grad))``.
    """
    assert px.ndim == 3
    B, S, T1 = px.shape
    T = py.shape[-1]
    assert px.shape[-1] in [T, T + 1]
    assert py.shape == (B, S + 1, T)
    assert px.dtype == py.dtype
    if boundary is not None:
        _assert_boundary(boundary, B, S, T, on_device=_lib.ops().deferred_checks())

    # one autograd node of the operator module (mutual_information.py:24-181): its forward runs
    # the forward operator and, when gradients may be needed, immediately the backward operator
    # with a gradient of ones; its backward only scales those stored occupation gradients (in
    # place, which also changes the tensors handed out here)
    scores, px_grad, py_grad = _lib.ops().recursion(px, py, boundary, bool(return_grad))
    return (scores, (px_grad, py_grad)) if return_grad else scores


def _inner_product(a: Tensor, b: Tensor) -> Tensor:
    """(a * b).sum(-1) with broadcasting, without the product as a temporary
    (fast_rnnt/python/fast_rnnt/mutual_information.py:301-311)."""
    assert a.shape[-1] == b.shape[-1]
    return torch.matmul(a.unsqueeze(-2), b.unsqueeze(-1)).squeeze(-1).squeeze(-1)


def joint_mutual_information_recursion(
    px: Sequence[Tensor], py: Sequence[Tensor], boundary: Optional[Tensor] = None,
) -> Sequence[Tensor]:
    """fast_rnnt/python/fast_rnnt/mutual_information.py:314-425.

    Runs the recursion on the sums ``sum(px)``, ``sum(py)`` and returns a tensor of
    shape ``(len(px), B)`` that splits the total score over the summands: term n gets
    the occupation-weighted sums ``<px_grad, px[n]> + <py_grad, py[n]>``, and what is
    left of the total (log-of-sum minus sum-of-log) is credited to term 0.  The
    occupations come from the two recursion kernels with a gradient of ones; they
    carry no autograd history, so the gradient of a share with respect to its own
    term is the occupation, as in the reference.
    """
    N = len(px)
    assert len(py) == N and N > 0
    B, S, T1 = px[0].shape
    T = py[0].shape[2]
    assert T1 in [T, T + 1]
    assert py[0].shape == (B, S + 1, T)
    assert px[0].dtype == py[0].dtype
    if boundary is not None:
        _assert_boundary(boundary, B, S, T, on_device=_lib.ops().deferred_checks())

    terms_x = torch.stack(tuple(px), dim=0)  # (N, B, S, T1)
    terms_y = torch.stack(tuple(py), dim=0)  # (N, B, S+1, T)
    with torch.no_grad():
        sum_x = terms_x.sum(dim=0).contiguous()
        sum_y = terms_y.sum(dim=0).contiguous()
        assert sum_x.ndim == 3 and sum_y.ndim == 3
        p = torch.empty(B, S + 1, T + 1, device=sum_x.device, dtype=sum_x.dtype)
        total = _fast_rnnt.mutual_information_forward(sum_x, sum_y, boundary, p)
        occ_x, occ_y = _fast_rnnt.mutual_information_backward(
            sum_x, sum_y, boundary, p, torch.ones(B, device=sum_x.device, dtype=sum_x.dtype))

    # a blocked cell (-inf) has occupation 0: raise it to a finite number so that the
    # product is 0, not nan (:411-412)
    floor = torch.finfo(terms_x.dtype).min
    shares = (_inner_product(occ_x.reshape(1, B, -1), terms_x.reshape(N, B, -1).clamp(min=floor))
              + _inner_product(occ_y.reshape(1, B, -1), terms_y.reshape(N, B, -1).clamp(min=floor)))
    with torch.no_grad():
        leftover = total - shares.sum(dim=0)
    shares[0] += leftover
    return shares
