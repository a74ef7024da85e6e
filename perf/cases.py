"""The calls that a training or evaluation program makes to this package, with the sizes it
makes them at, as cases that can be timed.

A case is one public function of the package on one batch: ``path`` names it, the sizes are
``B`` utterances of up to ``T`` encoder frames and ``S`` symbols over a vocabulary of ``C``,
``R`` kept symbol positions per frame for the pruned path.  Batches are ragged, as padded
batches of speech are: the first utterance has the full length and the others 0.6 - 1.0 of it.
``grad`` says whether the pass includes ``backward()``, as in training, or runs under
``no_grad``, as in validation.

float64 is left out: it serves gradient checks, not training.
"""
import math

import torch

import fast_rnnt_amd as F

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def _case(path, B, T, S, C, *, name=None, R=0, dtype="float32", rnnt_type="regular",
          reduction="sum", delay_penalty=0.0, lm_scale=0.0, am_scale=0.0, grad=True):
    case = dict(path=path, B=B, T=T, S=S, C=C, R=R, dtype=dtype, rnnt_type=rnnt_type,
                reduction=reduction, delay_penalty=delay_penalty, lm_scale=lm_scale,
                am_scale=am_scale, grad=grad)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # a few short utterances, as in a first trial, a unit test or the last batch of an epoch
        _case("simple", 4, 50, 10, 50, name="simple_smallest"),
        # the usual training step of a BPE-500 model
        _case("simple", 32, 250, 80, 500, name="simple_train"),
        # a batch filled up by duration on a card with much memory: longer utterances, more of them
        _case("simple", 64, 600, 120, 500, name="simple_large_batch"),
        # character-level vocabulary: the contraction over C is what counts
        _case("simple", 16, 400, 120, 5000, name="simple_large_vocab"),
        # under autocast: 2-byte inputs, odd sizes, the modified lattice with a delay penalty, as
        # streaming recipes train
        _case("simple", 21, 333, 47, 503, dtype="bfloat16", rnnt_type="modified",
              reduction="mean", delay_penalty=0.002, name="simple_bf16_modified_odd"),
        # first half of the pruned recipe: the smoothed loss and the pruning bounds from its
        # occupation gradients
        _case("smoothed", 32, 250, 80, 500, R=5, lm_scale=0.25, name="smoothed_and_ranges"),
        # between the two losses: pruning encoder and predictor outputs, and its backward
        _case("prune", 32, 250, 80, 500, R=5, name="prune_train"),
        # second half of the pruned recipe: the loss on the joiner's logits
        _case("pruned", 32, 250, 80, 500, R=5, name="pruned_train"),
        # the same under autocast with a character-level vocabulary
        _case("pruned", 16, 400, 120, 5000, R=5, dtype="bfloat16", name="pruned_bf16_large_vocab"),
        # the unpruned loss on the whole lattice of logits
        _case("joint", 8, 200, 60, 1000, name="joint_train"),
        # validation of a small unpruned model in half precision: forward only, a loss per utterance
        _case("joint", 5, 77, 19, 131, dtype="float16", reduction="none", grad=False,
              name="joint_fp16_validation"),
        # the lattice recursion on its own, on long utterances
        _case("recursion", 12, 1500, 220, 0, name="recursion_long"),
    ]


def _between(rng, low, high):
    """A whole number, spread evenly over the logarithm of [low, high]."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(["simple", "simple", "simple", "smoothed", "prune", "pruned", "pruned",
                       "joint", "recursion"])
    narrow = path in ("simple", "prune", "pruned", "joint") and rng.random() < 0.4
    dtype = rng.choice(["float16", "bfloat16"]) if narrow else "float32"
    rnnt_type = rng.choice(["regular", "regular", "regular", "modified", "constrained"])
    if path == "recursion" and rnnt_type == "constrained":
        rnnt_type = "modified"  # the recursion itself knows two kinds of lattice
    grad = path in ("smoothed", "prune") or rng.random() < 0.8
    C = _between(rng, 50, 5000)
    T = _between(rng, 40, 600 if path == "joint" else 1500)
    S = max(8, min(250, _between(rng, T / 12, T / 2.5)))
    R = rng.choice([3, 4, 5, 5, 5, 6, 8]) if path in ("smoothed", "prune", "pruned") else 0
    # batches are filled up to so many values of the largest tensor, the sum over a batch of
    # frames is what a program bounds, and no batch has more than 128 utterances
    row = {"simple": C, "smoothed": C, "prune": R * C, "pruned": R * C, "joint": (S + 1) * C,
           "recursion": S + 1}[path] * T
    limit = {"simple": 20e6, "smoothed": 10e6, "prune": 40e6, "pruned": 80e6, "joint": 80e6,
             "recursion": 4e6}[path]
    most = int(min(128, limit // row, 40000 // T))
    if most < 1:
        most, C = 1, max(50, int(C * limit / row))
    B = _between(rng, 1, most)
    if path == "recursion":
        C = 0
    return _case(path, B, T, S, C, R=R, dtype=dtype, rnnt_type=rnnt_type,
                 reduction=rng.choice(["sum", "sum", "mean"]) if grad else "none",
                 delay_penalty=rng.choice([0.0, 0.0, 0.002]) if path not in ("prune", "recursion")
                 else 0.0,
                 lm_scale=rng.choice([0.25, 0.1]) if path == "smoothed" else 0.0,
                 am_scale=rng.choice([0.0, 0.1]) if path == "smoothed" else 0.0, grad=grad)


def _lengths(case, g):
    """[B, 4] boundary rows [0, 0, S_b, T_b] of a padded batch."""
    B, T, S = case["B"], case["T"], case["S"]
    part = 0.6 + 0.4 * torch.rand(2, B, generator=g, device="cuda")
    part[:, 0] = 1.0
    t_end = (T * part[0]).round().long().clamp(min=1)
    s_end = torch.minimum((S * part[1]).round().long().clamp(min=1), t_end)
    zero = torch.zeros_like(t_end)
    return torch.stack([zero, zero, s_end, t_end], dim=1)


def _alignment(case, boundary):
    """[B, T]: the symbol position that a model which has learnt something is at in each frame."""
    t = torch.arange(case["T"], device="cuda")
    return torch.minimum(t * boundary[:, 2:3] // boundary[:, 3:4], boundary[:, 2:3] - 1)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    path, B, T, S, C, R = (case[k] for k in ("path", "B", "T", "S", "C", "R"))
    dtype = _DTYPES[case["dtype"]]
    boundary = _lengths(case, g)
    state = dict(case=case, boundary=boundary)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    def leaf(x):
        return x.to(dtype).requires_grad_(case["grad"])

    if path == "recursion":
        # log-probabilities of a symbol and of a blank in every cell
        T1 = T + 1 if case["rnnt_type"] == "regular" else T
        px = -3.0 + randn(B, S, T1)
        if T1 > T:
            px[:, :, T] = -math.inf
        state.update(px=leaf(px), py=leaf(-1.0 + 0.5 * randn(B, S + 1, T)))
        return state

    symbols = torch.randint(1, C, (B, S), generator=g, device="cuda")
    state["symbols"] = symbols
    at = _alignment(case, boundary)
    if path in ("simple", "smoothed", "prune"):
        # encoder and predictor outputs: noise, and a preference for blanks and, along the
        # alignment, for the symbol that is next
        am = (2.0 if C < 1000 else 1.0) * randn(B, T, C)
        lm = (2.0 if C < 1000 else 1.0) * randn(B, S + 1, C)
        am[:, :, 0] += 3.0
        am.scatter_add_(2, symbols.gather(1, at).unsqueeze(2), torch.full((B, T, 1), 3.0, device="cuda"))
        state.update(am=leaf(am), lm=leaf(lm))
    if path == "prune":
        # occupation probabilities as a smoothed loss leaves them: a band around the alignment
        with torch.no_grad():
            s = torch.arange(S + 1, device="cuda").reshape(1, S + 1, 1)
            band = torch.exp(-0.5 * ((s - at.unsqueeze(1)) / 1.5) ** 2)
            band = band * (0.5 + torch.rand(B, S + 1, T, generator=g, device="cuda"))
            py_grad = band / band.sum(dim=1, keepdim=True)
            T1 = T + 1 if case["rnnt_type"] == "regular" else T
            px_grad = torch.zeros(B, S, T1, device="cuda")
            px_grad[:, :, :T] = py_grad[:, :S] * (S / T)
        state.update(px_grad=px_grad, py_grad=py_grad,
                     upstream=randn(B, T, min(R, S + 1), C).to(dtype))
    if path == "pruned":
        # the bounds of a pruned lattice: R positions per frame, from the first to the last symbol
        t = torch.arange(T, device="cuda")
        room = (boundary[:, 2:3] + 1 - R).clamp(min=0)
        begin = torch.minimum(t * room // (boundary[:, 3:4] - 1).clamp(min=1), room)
        state["ranges"] = begin.unsqueeze(2) + torch.arange(R, device="cuda")
    if path in ("pruned", "joint"):
        logits = randn(B, T, R if path == "pruned" else S + 1, C)
        logits[..., 0] += 2.0
        state["logits"] = leaf(logits)
    return state


def run(state):
    case, boundary = state["case"], state["boundary"]
    path, grad = case["path"], case["grad"]
    kinds = dict(rnnt_type=case["rnnt_type"], delay_penalty=case["delay_penalty"],
                 reduction=case["reduction"])
    with torch.set_grad_enabled(grad):
        if path == "simple":
            am, lm = state["am"], state["lm"]
            am.grad = lm.grad = None
            loss, (px_grad, py_grad) = F.rnnt_loss_simple(
                lm, am, state["symbols"], 0, boundary=boundary, return_grad=True, **kinds)
            if not grad:
                return dict(loss=loss, px_grad=px_grad, py_grad=py_grad)
            loss.backward()
            return dict(loss=loss.detach(), px_grad=px_grad, py_grad=py_grad, am_grad=am.grad,
                        lm_grad=lm.grad)
        if path == "smoothed":
            am, lm = state["am"], state["lm"]
            am.grad = lm.grad = None
            loss, (px_grad, py_grad) = F.rnnt_loss_smoothed(
                lm, am, state["symbols"], 0, lm_only_scale=case["lm_scale"],
                am_only_scale=case["am_scale"], boundary=boundary, return_grad=True, **kinds)
            ranges = F.get_rnnt_prune_ranges(px_grad, py_grad, boundary, case["R"])
            loss.backward()
            return dict(loss=loss.detach(), ranges=ranges, px_grad=px_grad, py_grad=py_grad,
                        am_grad=am.grad, lm_grad=lm.grad)
        if path == "prune":
            am, lm = state["am"], state["lm"]
            am.grad = lm.grad = None
            ranges = F.get_rnnt_prune_ranges(state["px_grad"], state["py_grad"], boundary,
                                             case["R"])
            am_pruned, lm_pruned = F.do_rnnt_pruning(am, lm, ranges)
            # (the joiner that comes next adds the two, so both get the same gradient)
            torch.autograd.backward([am_pruned, lm_pruned], [state["upstream"]] * 2)
            return dict(ranges=ranges, lm_pruned=lm_pruned.detach(), am_grad=am.grad,
                        lm_grad=lm.grad)
        if path in ("pruned", "joint"):
            logits = state["logits"]
            logits.grad = None
            if path == "pruned":
                loss = F.rnnt_loss_pruned(logits, state["symbols"], state["ranges"], 0,
                                          boundary=boundary, **kinds)
            else:
                loss = F.rnnt_loss(logits, state["symbols"], 0, boundary=boundary, **kinds)
            if not grad:
                return dict(loss=loss)
            loss.backward()
            return dict(loss=loss.detach(), logits_grad=logits.grad)
        px, py = state["px"], state["py"]
        px.grad = py.grad = None
        if not grad:
            return dict(scores=F.mutual_information_recursion(px, py, boundary))
        scores = F.mutual_information_recursion(px, py, boundary)
        (-scores.sum()).backward()
        return dict(scores=scores.detach(), px_grad=px.grad, py_grad=py.grad)


def work(case):
    """Bytes and floating-point operations of one pass.  A batch's windows cover 0.8 of the frames
    and 0.8 of the symbols on average; what lies outside is not needed, but gradients are written
    whole, zeros included."""
    path, B, T, S, C, R = (case[k] for k in ("path", "B", "T", "S", "C", "R"))
    grad = case["grad"]
    item = torch.empty((), dtype=_DTYPES[case["dtype"]]).element_size()
    frames, rows, cells = 0.8 * B * T, 0.8 * B * (S + 1), 0.64 * B * T * (S + 1)
    lattice = 4 * B * (2 * S + 1) * T  # px_grad and py_grad
    labels = 8 * B * S + 32 * B
    if path in ("simple", "smoothed"):
        inputs = item * C * (frames + rows) + labels
        product = 2.0 * C * cells
        if not grad:
            return {"bytes": inputs + lattice, "flops": product}
        outputs = lattice + item * C * B * (T + S + 1) + 8 * B * T * R
        return {"bytes": inputs + outputs, "flops": 3 * product}
    if path == "prune":
        pruned = item * B * T * R * C
        both = item * C * B * (T + S + 1)
        return {"bytes": lattice + 8 * B * T * R + item * C * B * (S + 1) + 2 * pruned + both,
                "flops": 2.0 * B * T * R * C}
    if path in ("pruned", "joint"):
        read = (frames * R if path == "pruned" else cells) * C
        written = B * T * (R if path == "pruned" else S + 1) * C if grad else 0
        index = 8 * frames * R if path == "pruned" else 0
        return {"bytes": item * (read + written) + index + labels,
                "flops": (8.0 if grad else 4.0) * read}
    bytes_in = 4 * 2 * cells
    return {"bytes": bytes_in + (lattice if grad else 0) + 32 * B,
            "flops": (20.0 if grad else 10.0) * cells}


def tolerance(case):
    """Gradients are exponentials of differences of lattice scores.  A score is about two nats per
    step, several hundred to several thousand in all, and has a rounding error of 2^-24 of that:
    moving the log-probabilities of a lattice by one unit in the last place moves its occupation
    probabilities by 1e-5 - 3e-5 of their norm and by up to 3e-4 in single cells, and the steps
    of the recursion round once each.  2-byte gradients add the rounding of their type; pruning
    bounds are whole numbers that turn on which of two sums is larger."""
    if not case["grad"] and case["path"] != "simple":
        return {"rel": 1e-5, "max": 1e-4}  # the scores alone
    narrow = {"float32": 0.0, "float16": 1e-3, "bfloat16": 8e-3}[case["dtype"]]
    if case["path"] == "prune":
        # sums of R values of the input's type per frame, in torch's order for am
        return {"rel": max(1e-6, narrow), "max": max(1e-5, 4 * narrow)}
    tol = {"rel": max(1e-4, narrow), "max": max(2e-3, 4 * narrow)}
    if case["path"] == "smoothed":
        tol["differ"] = 2e-3
    return tol
