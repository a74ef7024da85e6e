"""The recursion where every band of 64 lattice rows has a workgroup of its own: two, three and four
bands, sizes at the edges of bands and of 32-step tiles, windows that leave bands out, are empty or
start inside the lattice.  The same utterances in a batch too large for that run with one workgroup
each: the results must be the same bits.  Oracle: the CPU restatement in float32."""
import pytest
import torch

from fast_rnnt_amd import _fast_rnnt, _lib
from oracle import recursion as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T", [(64, 1200), (100, 900), (127, 800), (128, 700), (129, 513), (191, 600),
                                 (192, 320), (200, 257), (255, 288), (255, 300)])
def test_bands_in_workgroups_of_their_own(gpu_device, S, T, modified):
    g = torch.Generator().manual_seed(S + T)
    rows = [[0, 0, S, T], [0, 0, S, T - 1], [0, 0, min(S, 63), T], [0, 0, 64, T], [1, 3, S, T],
            [2, 1, S - 1, T - 31], [0, 0, S, 0], [5, 9, 5, T], [0, 5, S // 2, T - 7]]
    n, T1 = len(rows), T if modified else T + 1
    px = -1 + torch.randn(n, S, T1, generator=g)
    py = -1 + torch.randn(n, S + 1, T, generator=g)
    bnd = torch.tensor(rows)

    def run(copies):
        args = [x.to(gpu_device).repeat(copies, 1, 1) for x in (px, py)]
        args.append(bnd.to(gpu_device).repeat(copies, 1))
        p = torch.zeros(n * copies, S + 1, T + 1, device=gpu_device)
        print(f"S={S} T={T} modified={modified} B={n * copies}", flush=True)
        scores = _fast_rnnt.mutual_information_forward(*args, p)
        seed = torch.ones(n * copies, device=gpu_device)
        gx, gy = _fast_rnnt.mutual_information_backward(*args, p, seed)
        return [x[-n:].cpu() for x in (scores, p, gx, gy, seed)]

    got, whole = run(1), run(30)
    for a, b in zip(got, whole):
        assert torch.equal(a, b)
    p_cpu = torch.zeros(n, S + 1, T + 1)
    want = oracle.mi_forward(px, py, bnd, p_cpu)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got[0]), finite)
    assert bool(((got[0] - want).abs()[finite] <= 1e-5 * want.abs()[finite].clamp(min=1)).all())
    gx, gy = oracle.mi_backward(px, py, bnd, p_cpu, torch.ones(n))
    for a, b in ((got[2], gx), (got[3], gy)):
        assert not torch.isnan(a).any() and bool((a - b).norm() <= 2e-3 * b.norm().clamp(min=1))


LONG = [(64, 12988), (65, 12989), (100, 13480), (255, 14000), (70, 30700), (250, 686), (192, 748),
        (255, 749), (150, 4074), (100, 10730)]


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T,dtype", [(*size, torch.float32) for size in LONG] +
                         [(100, 700, torch.float64), (100, 749, torch.float64),
                          (40, 10732, torch.float64)])
def test_every_length_finds_a_launch_that_fits(gpu_device, S, T, dtype, modified):
    """The LDS of a workgroup grows with T.  float32: a band has a workgroup to itself up to
    T = 12 988; a workgroup holds four sweep waves up to T = 748, three up to 4 076, two up to
    10 732, one up to 30 700.  float64: two up to 748, one up to 10 732."""
    g = torch.Generator().manual_seed(S + T)
    T1 = T if modified else T + 1
    px = -4 + torch.randn(1, S, T1, generator=g, dtype=dtype)
    py = -0.1 * torch.rand(1, S + 1, T, generator=g, dtype=dtype)
    print(f"S={S} T={T} {dtype} modified={modified}", flush=True)
    p = torch.zeros(1, S + 1, T + 1, device=gpu_device, dtype=dtype)
    x, y = px.to(gpu_device), py.to(gpu_device)
    score = _fast_rnnt.mutual_information_forward(x, y, None, p)
    gx, gy = _fast_rnnt.mutual_information_backward(x, y, None, p, torch.ones_like(score))
    want = oracle.mi_forward(px, py, None, torch.zeros(1, S + 1, T + 1, dtype=dtype))
    assert abs(score.item() - want.item()) <= 1e-5 * abs(want.item())
    # every path passes every frame once; each of the S + T steps of a path rounds once
    frames = gy.double().sum(1) + (gx.double().sum(1) if modified else 0)
    assert bool(((frames - 1).abs() <= (S + T) * 2.0 ** -24).all()), (frames - 1).abs().max().item()


@pytest.mark.parametrize("modified", [False, True])
@pytest.mark.parametrize("S,T", [(100, 900), (250, 700)])
def test_a_wait_that_runs_out_in_any_band_shows_as_nan(gpu_device, S, T, modified):
    """Whichever band's waits run out, the utterance's score is NaN, and so is a gradient of it and
    what reaches its start, unless every cell is what it is without a bound."""
    B, T1 = 8, T if modified else T + 1
    g = torch.Generator().manual_seed(S + T)
    px = (-1 + torch.randn(B, S, T1, generator=g)).to(gpu_device)
    py = (-1 + torch.randn(B, S + 1, T, generator=g)).to(gpu_device)

    def forward():
        p = torch.full((B, S + 1, T + 1), 12345.0, device=gpu_device)
        return _fast_rnnt.mutual_information_forward(px, py, None, p), p

    def backward():
        seed = torch.ones(B, device=gpu_device)
        return (*_fast_rnnt.mutual_information_backward(px, py, None, p, seed), seed)

    score, p = forward()
    gx, gy, seed = backward()
    lib = _lib.load()
    gave_up = 0
    for polls in (1, 2, 5, 20, 60, 150, 400, 1000, 1 << 22):
        print(f"S={S} T={T} modified={modified} polls={polls}", flush=True)
        lib.frnnt_set_spin_limit(polls)
        try:
            score1, p1 = forward()
            gx1, gy1, seed1 = backward()
            torch.cuda.synchronize()
        finally:
            lib.frnnt_set_spin_limit(0)
        for b in range(B):
            failed = bool(torch.isnan(score1[b]))
            gave_up += failed
            assert failed or (torch.equal(score1[b], score[b]) and torch.equal(p1[b], p[b]))
            nan = bool(torch.isnan(gx1[b]).any()), bool(torch.isnan(gy1[b]).any())
            if not any(nan) and not torch.isnan(seed1[b]):
                assert torch.equal(gx1[b], gx[b]) and torch.equal(gy1[b], gy[b])
                assert torch.equal(seed1[b], seed[b])
            else:
                assert all(nan) and bool(torch.isnan(seed1[b]))
        assert polls > 1 or gave_up == B
        assert polls < 1 << 22 or torch.equal(score1, score)
