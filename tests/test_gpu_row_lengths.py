"""The row kernels of the losses on logits (csrc/lattice_logprobs.hip, lattice_gradient.hip) where
their split of a row over lanes and 16-byte pieces can go wrong: vocabularies on either side of every
split (a quarter, a half, a whole wave per row, 2 ... 20 pieces per lane, rows in chunks), rows that
share a piece with their neighbours, logits that begin off a 16-byte boundary.  Oracle: the CPU
restatement on the same values in float32."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu
# gradients: 1e-4 absolute and one unit in the last place of the type
ULP = {torch.float32: 1e-5, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}
LENGTHS = [1, 3, 63, 64, 65, 125, 128, 131, 256, 257, 503, 1025, 2050, 2565, 3590, 5113, 5121,
           10245]


@pytest.mark.parametrize("C", LENGTHS)
@pytest.mark.parametrize("dtype", list(ULP))
def test_loss_on_logits_of_any_row_length(gpu_device, dtype, C):
    B, S, T, R = 2, 4, 9, 3
    g = torch.Generator().manual_seed(C)
    symbols = torch.randint(0, C, (B, S), generator=g)
    boundary = torch.tensor([[0, 0, S, T], [0, 1, S - 1, T - 2]])
    begin = torch.clamp(torch.arange(T) * (S + 1 - R) // (T - 3), max=S + 1 - R)
    ranges = (begin.reshape(1, T, 1) + torch.arange(R)).expand(B, T, R).contiguous()
    for ranges_, K, shift, kind, handed_out in [(None, S + 1, 0, "regular", True),
                                                (None, S + 1, 1, "constrained", False),
                                                (ranges, R, 0, "modified", False),
                                                (ranges, R, 3, "regular", False)]:
        print(f"C={C} {dtype} K={K} shift={shift} {kind}", flush=True)
        flat = (2 * torch.randn(shift + B * T * K * C, generator=g)).to(dtype)
        cpu = flat[shift:].reshape(B, T, K, C).float().requires_grad_(True)
        gpu = flat.to(gpu_device)[shift:].reshape(B, T, K, C).requires_grad_(True)
        args = dict(boundary=boundary, rnnt_type=kind, delay_penalty=0.01, reduction="mean")
        dev = dict(args, boundary=boundary.to(gpu_device), return_grad=handed_out)
        if ranges_ is None:
            want = O.loss_joint(cpu, symbols, 0, **args)
            got = fast_rnnt_amd.rnnt_loss(gpu, symbols.to(gpu_device), 0, **dev)
        else:
            want = O.loss_pruned(cpu, symbols, ranges_, 0, **args)
            got = fast_rnnt_amd.rnnt_loss_pruned(gpu, symbols.to(gpu_device),
                                                 ranges_.to(gpu_device), 0, **dev)
        got = got[0] if handed_out else got
        assert abs(got.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
        (3.0 * want).backward()
        (3.0 * got).backward()
        off = (gpu.grad.float().cpu() - cpu.grad).abs()
        assert bool((off <= 1e-4 + ULP[dtype] * cpu.grad.abs()).all()), off.max().item()


# vocabularies (in 16-byte pieces) on either side of every split of a row
PIECES = [1, 15, 16, 17, 32, 33, 64, 65, 128, 129, 192, 193, 256, 257, 384, 385, 512, 513, 640, 641,
          896, 897, 1280, 1281]


@pytest.mark.parametrize("sfx,dtype", [("f32", torch.float32), ("f16", torch.float16),
                                       ("bf16", torch.bfloat16)])
def test_gradients_of_aligned_rows_are_the_bits_of_any_others(gpu_device, sfx, dtype):
    # the same rows through the kernel for rows that begin and end on 16 bytes, the one for any
    # alignment (logits and gradients one element off) and the one without pieces (one of them off)
    from fast_rnnt_amd import _lib
    B, S, T, R = 2, 5, 6, 3
    g = torch.Generator().manual_seed(9)
    T1 = T + 1
    symbols = torch.randint(0, 4, (B, S), generator=g).to(gpu_device)
    boundary = torch.tensor([[0, 0, S, T], [0, 1, S - 1, T - 1]]).to(gpu_device)
    ranges = (torch.tensor([0, 0, 1, 2, 3, 3]).reshape(1, T, 1) + torch.arange(R)).expand(B, T, R)
    ranges = ranges.contiguous().to(gpu_device)
    gx = torch.rand(B, S, T1, generator=g).to(gpu_device)
    gy = torch.rand(B, S + 1, T, generator=g).to(gpu_device)
    for pieces in PIECES:
        C = pieces * (16 // dtype.itemsize)
        n = B * T * R * C
        values = (2 * torch.randn(n, generator=g)).to(dtype).to(gpu_device)
        norm = torch.logsumexp(values.reshape(B * T * R, C).float(), 1)
        results = []
        for in_off, out_off in ((0, 0), (1, 1), (1, 0)):
            print(f"{dtype} C={C} offsets {in_off} {out_off}", flush=True)
            logits = torch.zeros(n + 8, dtype=dtype, device=gpu_device)
            logits[in_off:in_off + n] = values
            out = torch.full((n + 8,), 7.0, dtype=dtype, device=gpu_device)
            _lib.call("frnnt_lattice_logprobs_bwd_" + sfx, logits[in_off:].data_ptr(),
                      symbols.data_ptr(), ranges.data_ptr(), boundary.data_ptr(), norm.data_ptr(),
                      gx.data_ptr(), gy.data_ptr(), out[out_off:].data_ptr(), B, S, T, R, C, 3, 0, 1,
                      _lib.stream_of(out))
            assert bool((out[:out_off] == 7).all()) and bool((out[out_off + n:] == 7).all())
            results.append(out[out_off:out_off + n])
        assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])


@pytest.mark.parametrize("B,C", [(3, 750), (12, 751), (16, 752)])
def test_streamed_logits_give_the_bits_of_their_utterances(gpu_device, B, C):
    # 105, 419 and 560 MiB: past the sizes from which the gradient, a forward pass alone and a forward pass
    # before a backward are streamed; an utterance alone takes none of these paths
    T, S = 200, 60
    g = torch.Generator(device=gpu_device).manual_seed(C)
    logits = torch.randn(B, T, S + 1, C, generator=g, device=gpu_device)
    symbols = torch.randint(1, C, (B, S), generator=g, device=gpu_device)
    ends = torch.tensor([[0, 0, S - 5 * (b % 3), T - 17 * (b % 4)] for b in range(B)], device=gpu_device)

    def run(rows):
        leaf = logits[rows].clone().requires_grad_(True)
        loss = fast_rnnt_amd.rnnt_loss(leaf, symbols[rows], 0, boundary=ends[rows], reduction="none")
        loss.sum().backward()
        return loss.detach(), leaf.grad

    loss, grad = run(slice(0, B))
    with torch.no_grad():  # (the forward that no backward follows has a line of its own)
        alone = fast_rnnt_amd.rnnt_loss(logits, symbols, 0, boundary=ends, reduction="none")
    assert torch.equal(alone, loss)
    for b in range(B):
        one_loss, one_grad = run(slice(b, b + 1))
        assert torch.equal(loss[b:b + 1], one_loss) and torch.equal(grad[b:b + 1], one_grad)
