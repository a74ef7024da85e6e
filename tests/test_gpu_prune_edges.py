"""The kernels behind get_rnnt_prune_ranges at the edges of their splits: frame counts around a tile of 32 and
around one run of frames per thread (256) and per batch of loads (1024), candidate starts around four and eight per
group of sixteen, windows of 1 to 17 (plain and cascaded sums).  Bit-exact against the oracle."""
import pytest
import torch

import fast_rnnt_amd
from oracle import losses as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("S,T", [(1, 1), (2, 31), (9, 33), (17, 255), (18, 256), (33, 257), (63, 32), (65, 96), (127, 64), (128, 65),
                                 (129, 66), (130, 1023), (5, 1024), (6, 1025), (40, 2600)])
def test_ranges_at_the_edges_of_the_splits(gpu_device, S, T, dtype):
    B, g = 3, torch.Generator().manual_seed(S + T)
    Tb = torch.randint(max(1, T // 2), T + 1, (B,), generator=g)
    Sb = torch.minimum(torch.randint(max(1, S // 2), S + 1, (B,), generator=g), Tb)
    z = torch.zeros(B, dtype=torch.int64)
    bnd = torch.stack([z, z, Sb, Tb], 1)
    for kind, T1 in (("regular", T + 1), ("modified", T)):
        gx, gy = (torch.rand(B, S, T1, generator=g, dtype=dtype), torch.rand(B, S + 1, T, generator=g, dtype=dtype))
        gy[0, :, ::3] = (4 * gy[0, :, ::3]).round() / 4  # (ties)
        for R in (2, 3, 8, 16, 17):
            if R > S + 1:
                continue
            want = O.prune_ranges(gx, gy, bnd, R, **({"window_sum": "cascade"} if R > 16 else {}))
            got = fast_rnnt_amd.get_rnnt_prune_ranges(gx.to(gpu_device), gy.to(gpu_device), bnd.to(gpu_device), R)
            assert torch.equal(got.cpu(), want)
