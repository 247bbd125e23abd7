"""The alpha statistics kernels (muzero_block_stats, muzero_select3) against the torch formulation they
replace, bit for bit: types, head dims, short and long blocks, strided storage, non-finite values, and
subsamples of one value up to more than one chunk of the selection."""

import math

import pytest
import torch

from muzero_amd import quantizer as Q
from muzero_amd.kernels import loader as L

pytestmark = pytest.mark.gpu


def _torch_statistics(block, kind, max_points):
    """The reference's statistics of the materialized rows, on the device (quantizer.py:46-55)."""
    b, h, t, d = block.shape
    rows = block.reshape(b, h, t // 64, 64, d).transpose(3, 4).reshape(-1, 64) if kind == "key" else block.reshape(-1, 64)
    lo, hi = rows.float().amin(-1), rows.float().amax(-1)
    za = ((0.0 - lo) / (hi - lo).clamp_min(1e-8)).clamp(0.0, 1.0)
    flat = Q._subsample(rows, max_points).float().abs()
    srt = torch.sort(flat).values
    mean = (za - 0.5).abs().reshape(1, 1, 1, -1).mean()
    return torch.stack([*(srt[k] for k in Q._percentile_ranks(flat.numel())), mean]).tolist()


@pytest.mark.parametrize("kind", ["key", "value"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape,max_points", [((1, 1, 64, 64), 65536), ((2, 3, 128, 192), 1000), ((3, 8, 1984, 128), 65536),
                                              ((2, 4, 640, 128), 200_000), ((1, 2, 64, 320), 1)])
def test_block_statistics(kind, dtype, shape, max_points):
    b, h, t, d = shape
    g = torch.Generator().manual_seed(t + d)
    cap = torch.randn(b, h, t + 72, d, generator=g)
    cap[..., :3] *= 10
    block = cap.to(dtype).cuda()[:, :, 8:8 + t]
    assert Q._kernel_statistics(block, 64, kind, max_points)
    got = Q._block_statistics(block, 64, kind, max_points)
    assert got == _torch_statistics(block, kind, max_points)
    both = Q.select_alpha_blocks({"key": block, "value": block}, bits=8, q_group_size=64, max_points=max_points)
    assert both == {k: Q.select_alpha_block(block, bits=8, q_group_size=64, kind=k, max_points=max_points) for k in both}


@pytest.mark.parametrize("kind", ["key", "value"])
def test_non_finite_blocks(kind):
    block = torch.randn(2, 2, 256, 128, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    block[0, 0, 5, 3], block[1, 1, 200, 64], block[0, 1, 70, 9] = float("nan"), float("inf"), float("-inf")
    for value in (block, torch.zeros_like(block), torch.full_like(block, float("nan"))):
        got = Q._block_statistics(value.cuda(), 64, kind, 65536)
        want = _torch_statistics(value.cuda(), kind, 65536)
        assert all(x == y or (math.isnan(x) and math.isnan(y)) for x, y in zip(got, want)), (got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 3, 64, 4095, 4097, 32768, 65537, 100_003])
def test_select(n, dtype):
    g = torch.Generator().manual_seed(n)
    x = torch.rand(n, generator=g) * torch.logspace(-30, 30, n)
    x[::7] = 1.5  # ties
    x = x[torch.randperm(n, generator=g)].to(dtype).cuda()
    ranks = [0, n // 2, n - 1]
    two = torch.zeros(2, (n + 7) // 8 * 8, device="cuda", dtype=dtype)
    two[0, :n], two[1, :n] = x, x.flip(0) * 3
    out = torch.empty(2, 3, device="cuda")
    L.check(L.load().muzero_select3(two.data_ptr(), L.DTYPE_ENUM[dtype], 2, two.stride(0), n, *ranks, out.data_ptr(), 3,
                                    L.stream_ptr(x.device)), "select")
    assert out.tolist() == [[torch.sort(row).values[k].item() for k in ranks] for row in two[:, :n]]
