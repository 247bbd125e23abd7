"""The bf16 and fp16 quantize kernels on the magnitudes where their path changes (GPU), bit for bit
against the oracle, at each width.  bf16: values around 2^121 (from there a bf16 pattern read as fp16 is
infinite and its group takes the general chain), scales around 2^126 (the reciprocal of a larger one is
denormal), subnormals, zeros of both signs, every finite magnitude in one group.  fp16: subnormals (exact
ties of the quotients there), ordinary and largest magnitudes."""

import numpy as np
import pytest
import torch

from conftest import bits_of
from oracle import reference_torch as ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _patterns(lo, hi, shape, seed):
    """bf16 values of random sign and significand, exponent fields lo..hi."""
    g = torch.Generator().manual_seed(seed)
    u = (torch.randint(0, 2, shape, generator=g) << 15) | (torch.randint(lo, hi + 1, shape, generator=g) << 7)
    u = u | torch.randint(0, 128, shape, generator=g)
    return torch.where(u >= 32768, u - 65536, u).to(torch.int16).view(torch.bfloat16)


@pytest.mark.parametrize("lo, hi", [(0, 0), (0, 3), (120, 130), (246, 248), (252, 253), (0, 253)],
                         ids=["subnormal", "tiny", "ordinary", "edge121", "edge126", "all"])
@pytest.mark.parametrize("bits", range(1, 9))
def test_magnitude_edges_match_oracle(bits, lo, hi):
    x = _patterns(lo, hi, (1, 2, 128, 128), 10 * bits + lo)
    x[:, :, ::5] *= torch.tensor([0.0, 1.0], dtype=torch.bfloat16).repeat(64)
    _check(x, bits)


@pytest.mark.parametrize("step, span", [(2.0 ** -24, 20), (2.0 ** -24, 2000), (2.0 ** -10, 3000), (16.0, 2000)],
                         ids=["subnormal", "tiny", "ordinary", "largest"])
@pytest.mark.parametrize("bits", range(1, 9))
def test_fp16_magnitude_edges_match_oracle(bits, step, span):
    g = torch.Generator().manual_seed(bits)
    x = (torch.randint(-span, span + 1, (1, 2, 128, 128), generator=g) * step).to(torch.float16)
    _check(x, bits)


def _check(x, bits):
    from muzero_amd.kernels import loader as L
    b, h, t, d = x.shape
    qb, dx, meta = 8 * bits, x.to(DEV), torch.float32
    pk = torch.empty((b, h, t // 64, d, qb), dtype=torch.uint8, device=DEV)
    kmn = torch.empty((b, h, t // 64, d, 1), dtype=meta, device=DEV)
    ksc = torch.empty_like(kmn)
    L.quantize_key_block_into(dx, bits, 2.0, 1e-8, pk, kmn, ksc)
    pv = torch.empty((b, h, t, d // 64, qb), dtype=torch.uint8, device=DEV)
    vmn = torch.empty((b, h, t, d // 64, 1), dtype=meta, device=DEV)
    vsc = torch.empty_like(vmn)
    L.quantize_value_block_into(dx, bits, 2.0, 1e-8, pv, vmn, vsc)
    for got, want in zip((pk, kmn, ksc, pv, vmn, vsc), ref.quantize_key_block(x, bits, 2.0, 64, amax_dtype=meta)
                         + ref.quantize_value_block(x, bits, 2.0, 64, amax_dtype=meta)):
        if got.dtype == torch.uint8:
            np.testing.assert_array_equal(got.cpu().numpy(), want.numpy())
        else:
            np.testing.assert_array_equal(bits_of(got), bits_of(want))
