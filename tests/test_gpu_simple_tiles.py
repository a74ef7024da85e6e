"""rnnt_loss_simple where the kernels' choice of tiles and their splits into chunks can go wrong:
sizes on either side of a tile of lattice rows, frames and vocabulary entries, sums over few and
many chunks, batches small and large, 2-byte inputs, long lists of equal symbols.  Oracle: the CPU
restatement on the same values in float32."""
import ctypes

import pytest
import torch

import fast_rnnt_amd
from fast_rnnt_amd import _lib
from oracle import losses as O

pytestmark = pytest.mark.gpu
# (B, S, T, C)
SIZES = [(1, 1, 1, 1), (2, 1, 3, 31), (1, 31, 33, 32), (2, 32, 64, 33), (3, 63, 65, 64),
         (1, 64, 64, 65), (2, 95, 96, 129), (1, 127, 129, 300), (2, 128, 140, 70),
         (1, 20, 40, 4097), (2, 60, 70, 2600), (1, 130, 260, 1700), (5, 100, 190, 2050),
         (40, 70, 300, 40), (70, 33, 130, 130), (30, 130, 280, 66)]


@pytest.mark.parametrize("B,S,T,C", SIZES)
def test_simple_loss_at_the_edges_of_tiles(gpu_device, B, S, T, C):
    g = torch.Generator().manual_seed(B + S + T + C)
    t_end = (T * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1)
    s_end = torch.minimum((S * (0.6 + 0.4 * torch.rand(B, generator=g))).long().clamp(min=1), t_end)
    t_end[0], s_end[0] = T, min(S, T)
    zero = torch.zeros_like(t_end)
    boundary = torch.stack([zero, zero, s_end, t_end], 1)
    symbols = torch.randint(0, C, (B, S), generator=g)
    symbols[0] = C // 2  # every lattice row of an utterance on one vocabulary entry
    for dtype, kind in [(torch.float32, "regular"), (torch.bfloat16, "modified"),
                        (torch.float16, "constrained")]:
        print(f"B={B} S={S} T={T} C={C} {dtype} {kind}", flush=True)
        lm = (2 * torch.randn(B, S + 1, C, generator=g)).to(dtype)
        am = (2 * torch.randn(B, T, C, generator=g)).to(dtype)
        cpu = [x.float().clone().requires_grad_(True) for x in (lm, am)]
        gpu = [x.to(gpu_device).requires_grad_(True) for x in (lm, am)]
        args = dict(rnnt_type=kind, delay_penalty=0.01, reduction="mean")
        want = O.loss_simple(*cpu, symbols, 0, boundary=boundary, **args)
        got, occupation = fast_rnnt_amd.rnnt_loss_simple(
            *gpu, symbols.to(gpu_device), 0, boundary=boundary.to(gpu_device), return_grad=True,
            **args)
        assert abs(got.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
        (3.0 * want).backward()
        (3.0 * got).backward()
        assert occupation[0].dtype == torch.float32
        ulp = {torch.float32: 1e-4, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
        for x, y in zip(gpu, cpu):
            assert x.grad.dtype == dtype
            off = (x.grad.float().cpu() - y.grad).abs()
            assert bool((off <= 2e-4 + ulp * y.grad.abs()).all()), off.max().item()


def logprobs(lm, am, symbols, boundary, window_only):
    """px, py, lm_max, am_max and norm_raw of the regular lattice; NaN where nothing was written."""
    (B, S1, C), T = lm.shape, am.shape[1]
    shapes = [(B, S1 - 1, T + 1), (B, S1, T), (B, S1), (B, T), (B, S1, T)]
    out = [torch.full(n, float("nan"), device=lm.device) for n in shapes]
    _lib.call("frnnt_simple_logprobs_fwd_f32", lm.data_ptr(), am.data_ptr(), symbols.data_ptr(),
              _lib.ptr(boundary), *(x.data_ptr() for x in out), B, S1 - 1, T, C, 0, 0, window_only,
              _lib.stream_of(am))
    return out


# (B, S, T, C): fewer and more tiles than compute units, one, two and more waves' lanes of utterances,
# short and long loops (the product takes eight or four waves, and the four have one, two, four and
# five slabs of a share), one row of 384 and 650 tiles
WINDOWED = [(3, 40, 70, 33), (9, 200, 300, 700), (64, 63, 65, 90), (65, 31, 200, 40),
            (130, 64, 129, 20), (300, 5, 33, 9), (40, 33, 256, 1100),
            (96, 14, 114, 300), (130, 31, 150, 300), (30, 40, 250, 300), (15, 63, 450, 400),
            (16, 90, 500, 300), (30, 130, 280, 500), (28, 127, 250, 640)]


@pytest.mark.parametrize("B,S,T,C", WINDOWED)
def test_tiles_of_windows_are_the_tiles_of_the_whole_lattice(gpu_device, B, S, T, C):
    # the tiles that count are found from the windows of the whole batch; each must be there, and hold
    # the bits that the whole lattice has there
    g = torch.Generator().manual_seed(B + S)
    edges_s = torch.tensor([0, 1, 30, 31, 32, 62, 63, 64, S - 1, S]).clamp(max=S)
    edges_t = torch.tensor([0, 1, 31, 32, 33, 64, T - 1, T]).clamp(max=T)
    s_end = edges_s[torch.randint(len(edges_s), (B,), generator=g)]
    t_end = edges_t[torch.randint(len(edges_t), (B,), generator=g)]
    s_end[B // 2], t_end[B // 2] = S, T
    boundary = torch.stack([torch.zeros_like(s_end)] * 2 + [s_end, t_end], 1).to(gpu_device)
    lm = torch.randn(B, S + 1, C, generator=g).to(gpu_device)
    am = torch.randn(B, T, C, generator=g).to(gpu_device)
    symbols = torch.randint(0, C, (B, S), generator=g).to(gpu_device)

    whole, windowed = (logprobs(lm, am, symbols, boundary, w) for w in (0, 1))
    s = torch.arange(S + 1, device=gpu_device).view(1, -1, 1)
    t = torch.arange(T + 1, device=gpu_device).view(1, 1, -1)
    rows, frames = s <= boundary[:, 2].view(-1, 1, 1), t < boundary[:, 3].view(-1, 1, 1)
    last = t <= boundary[:, 3].view(-1, 1, 1)  # (the -inf that closes the lattice)
    px_there = (rows[:, :S] & last) | (t == T)
    there = [px_there, rows & frames[:, :, :T], rows[:, :, 0], frames[:, 0, :T],
             rows & frames[:, :, :T]]
    for got, want, here in zip(windowed, whole, there):
        assert not torch.isnan(want).any()
        assert torch.equal(got[here], want[here])


# (S, T, C, s_end, t_end): sums over k that end before, at and after a chunk of 32 and a k-step of 16,
# rows of D whose length is no multiple of 4, lists of 16, 17, 128 and more equal symbols
CHUNKS = [(16, 33, 70, 15, 31), (17, 34, 70, 16, 32), (40, 61, 65, 31, 33), (33, 255, 64, 32, 47),
          (70, 98, 130, 63, 64), (140, 257, 66, 128, 65), (145, 150, 64, 145, 150)]


@pytest.mark.parametrize("S,T,C,s_end,t_end", CHUNKS)
def test_gradient_products_read_nothing_outside_a_window(gpu_device, S, T, C, s_end, t_end):
    g = torch.Generator().manual_seed(S + T)
    lm, am = torch.randn(2, S + 1, C, generator=g), torch.randn(2, T, C, generator=g)
    symbols = torch.full((2, S), C // 2)
    boundary = torch.tensor([[0, 0, s_end, t_end], [0, 0, s_end - 1, t_end - 1]])
    cpu = [x.clone().requires_grad_(True) for x in (lm, am)]
    O.loss_simple(*cpu, symbols, 0, boundary=boundary, reduction="sum").backward()
    for b in range(2):  # rows and frames outside the windows must not be looked at
        lm[b, boundary[b, 2] + 1:] = float("nan")
        am[b, boundary[b, 3]:] = float("nan")
    gpu = [x.to(gpu_device).requires_grad_(True) for x in (lm, am)]
    loss = fast_rnnt_amd.rnnt_loss_simple(*gpu, symbols.to(gpu_device), 0,
                                          boundary=boundary.to(gpu_device), reduction="sum")
    # (what the scratch of the backward holds before it runs)
    del_me = [torch.full((n,), float("nan"), device=gpu_device) for n in (1 << 10, 1 << 14, 1 << 18)]
    del del_me
    loss.backward()
    for x, y in zip(gpu, cpu):
        assert bool(((x.grad.cpu() - y.grad).abs() <= 2e-4 + 1e-4 * y.grad.abs()).all())


# (S, T, C, [(B, whether with windows, rows of a tile, waves that share it)]): every form of the product
HEIGHTS = [(95, 128, 500, [(1, 0, 32, 8), (26, 0, 64, 8), (51, 0, 96, 8), (70, 0, 32, 4),
                           (26, 1, 64, 8), (40, 1, 32, 8), (64, 1, 96, 8), (70, 1, 32, 4)]),
           (120, 200, 600, [(1, 0, 32, 8), (11, 0, 64, 8), (22, 0, 32, 4), (37, 0, 32, 4),
                            (16, 1, 64, 8), (20, 1, 32, 8), (37, 1, 32, 4)])]


@pytest.mark.parametrize("S,T,C,batches", HEIGHTS)
def test_normalizers_are_the_same_bits_in_tiles_of_any_height(gpu_device, S, T, C, batches):
    # some rows have values far above what their first entries suggest, so that their shifts are
    # raised on the way; their neighbours in a tile, which differ with its height, must not notice
    g = torch.Generator().manual_seed(S)
    most = max(B for B, *_ in batches)
    lm, am = torch.randn(most, S + 1, C, generator=g), torch.randn(most, T, C, generator=g)
    for x in (lm, am):
        for b, r in torch.nonzero(torch.rand(x.shape[:2], generator=g) < 0.05).tolist():
            x[b, r, torch.randint(C // 3, C, (3,), generator=g)] += 40.0
    symbols = torch.randint(0, C, (most, S), generator=g)
    # (the first utterance is whole, the others' windows end anywhere)
    s_end, t_end = torch.randint(1, S + 1, (most,), generator=g), torch.randint(1, T + 1, (most,), generator=g)
    s_end[0], t_end[0] = S, T
    boundary = torch.stack([torch.zeros_like(s_end)] * 2 + [s_end, t_end], 1).to(gpu_device)
    lm, am, symbols = lm.to(gpu_device), am.to(gpu_device), symbols.to(gpu_device)
    first = None
    for B, windowed, rows, waves in batches:
        print(f"S={S} T={T} C={C} B={B} windows={windowed}", flush=True)
        got_waves = ctypes.c_int()
        assert _lib.load().frnnt_simple_logprobs_tile(B, S, T, C, windowed, ctypes.byref(got_waves)) == rows
        assert got_waves.value == waves
        out = logprobs(lm[:B], am[:B], symbols[:B], boundary[:B] if windowed else None, windowed)
        if first is None:
            first = [x[0].clone() for x in out]
        for got, want in zip(out, first):
            assert torch.equal(got[0], want)
    # (the last column is closed)
    px, py = first[0][:, :T].double().cpu(), first[1].double().cpu()
    joint = lm[0].double().cpu().unsqueeze(1) + am[0].double().cpu().unsqueeze(0)  # [S+1][T][C]
    norm = torch.logsumexp(joint, dim=2)
    want_y = joint[:, :, 0] - norm
    want_x = joint[:S].gather(2, symbols[0].cpu().reshape(S, 1, 1).expand(S, T, 1)).squeeze(2) - norm[:S]
    for got, want in ((px, want_x), (py, want_y)):
        assert bool(((got - want).abs() <= 2e-6 * want.abs().clamp(min=1) + 2e-5).all())


def test_gradients_that_are_streamed_past_the_cache(gpu_device):
    # lm, am and their gradients take 278 MB together, more than the last-level cache: the gradients
    # are stored with another hint than those of the two halves of the batch
    B, S, T, C = 14, 120, 400, 5000
    g = torch.Generator(device=gpu_device).manual_seed(2)
    lm = torch.randn(B, S + 1, C, generator=g, device=gpu_device)
    am = torch.randn(B, T, C, generator=g, device=gpu_device)
    symbols = torch.randint(1, C, (B, S), generator=g, device=gpu_device)

    def grads(rows):
        leaves = [x[rows].clone().requires_grad_(True) for x in (lm, am)]
        fast_rnnt_amd.rnnt_loss_simple(*leaves, symbols[rows], 0, reduction="sum").backward()
        return [x.grad for x in leaves]

    whole, halves = grads(slice(0, B)), [grads(slice(0, 7)), grads(slice(7, B))]
    for i in range(2):
        assert torch.equal(whole[i], torch.cat([h[i] for h in halves]))
