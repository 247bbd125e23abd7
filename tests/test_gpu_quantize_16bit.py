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


@pytest.mark.parametrize("d, pitch", [(33, 33), (100, 100), (128, 129), (264, 264)],
                         ids=["odd", "partial", "misaligned", "wide"])
@pytest.mark.parametrize("bits", [1, 3, 4, 8])
@pytest.mark.parametrize("dtype, lo, hi", [(torch.bfloat16, 120, 130), (torch.bfloat16, 0, 3), (torch.bfloat16, 0, 255),
                                           (torch.float16, 120, 130), (torch.float16, 104, 150)])
def test_rows_read_value_by_value_match_oracle(dtype, lo, hi, bits, d, pitch):
    """Head dims and row pitches without 16-byte vectors, or too wide for the staged key tile; magnitudes around
    one, subnormal ones, and all there are with infinities and NaN (fp16 from 2^-23, so that no value becomes a
    zero: which of two zeros of opposite sign is the smaller one is not defined)."""
    x = _patterns(lo, hi, (1, 2, 128, d), bits + d).to(dtype)
    x[..., 1] = 0.25  # a constant key group
    _check(x, bits, pitch)


def test_every_significand_pair_of_minimum_and_value():
    """v - min for every pair of bf16 significands, 0 to 18 binades apart either way, of equal and opposite signs,
    in both halves of a dword.  Groups of one minimum and 63 neighbouring values lie near their largest, where at
    8 bits and an almost linear compander neighbouring bf16 quotients have different codes."""
    value = lambda sign, exponent, frac: (sign << 15) | ((127 + exponent) << 7) | frac
    groups = []
    for distance in range(-18, 19):
        for v_sign in (0, 1):
            for a in range(128):
                v = [value(v_sign, max(distance, 0), f) for f in range(128)]
                for first in (0, 63, 65):  # 63 values each
                    group = [value(1, max(-distance, 0), a)] + v[first:first + 63]
                    shift = a + first // 63
                    groups.append(group[shift % 64:] + group[:shift % 64])
    u = torch.tensor(groups)
    x = torch.where(u >= 32768, u - 65536, u).to(torch.int16).view(torch.bfloat16)
    x = torch.cat([x, -x.flip(0)])  # positive minima too
    assert x.shape[0] % 64 == 0
    _check(x[None, None], 8, alpha=0.02)


def _check(x, bits, pitch=None, alpha=2.0):
    from muzero_amd.kernels import loader as L
    b, h, t, d = x.shape
    qb, dx, meta = 8 * bits, x.to(DEV), torch.float32
    if pitch:
        dx = torch.empty((b, h, t, pitch), dtype=x.dtype, device=DEV)[..., :d].copy_(dx)
    pk = torch.empty((b, h, t // 64, d, qb), dtype=torch.uint8, device=DEV)
    kmn = torch.empty((b, h, t // 64, d, 1), dtype=meta, device=DEV)
    ksc = torch.empty_like(kmn)
    L.quantize_key_block_into(dx, bits, alpha, 1e-8, pk, kmn, ksc)
    pv = torch.empty((b, h, t, -(-d // 64), qb), dtype=torch.uint8, device=DEV)
    vmn = torch.empty((b, h, t, -(-d // 64), 1), dtype=meta, device=DEV)
    vsc = torch.empty_like(vmn)
    L.quantize_value_block_into(dx, bits, alpha, 1e-8, pv, vmn, vsc)
    for got, want in zip((pk, kmn, ksc, pv, vmn, vsc), ref.quantize_key_block(x, bits, alpha, 64, amax_dtype=meta)
                         + ref.quantize_value_block(x, bits, alpha, 64, amax_dtype=meta)):
        if got.dtype == torch.uint8:
            np.testing.assert_array_equal(got.cpu().numpy(), want.numpy())
        else:  # a NaN's sign and payload are the arithmetic unit's choice: by place
            got, nan = got.cpu(), torch.isnan(want)
            assert torch.equal(torch.isnan(got), nan)
            np.testing.assert_array_equal(bits_of(got.masked_fill(nan, 0)), bits_of(want.masked_fill(nan, 0)))
