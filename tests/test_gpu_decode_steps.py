"""Decode steps that re-use the launch arguments cached on a layer, each with another query, mask and length, against
the same step with new arguments, bit for bit: the fused kernels and the unfused path, through flushes (the prefix
grows, the residual shrinks) and a move of the residual window."""

import pytest
import torch

import muzero_amd as mz
from muzero_amd.cache.layer import MuZeroCacheLayer

pytestmark = pytest.mark.gpu
BF, F16 = torch.bfloat16, torch.float16


class _Module:
    num_key_value_groups = 2


def _mask(kind, tokens, dtype, g):
    if kind == "none":
        return None
    keep = torch.arange(tokens + 3, device="cuda") >= torch.randint(0, tokens // 2, (3, 1), generator=g, device="cuda")
    keep = keep[:, None, None]  # (three columns past the cache's end, as static masks have)
    return keep if kind == "bool" else torch.zeros(keep.shape, dtype=dtype, device="cuda").masked_fill(
        ~keep, torch.finfo(dtype).min)


@pytest.mark.parametrize("mask", ["none", "additive", "bool", "mixed"])
@pytest.mark.parametrize("d,bits,dtype,kernel", [(128, 4, BF, "codebook"), (64, 4, F16, "fold"), (128, 8, BF, "twopass"),
                                                 (96, 4, BF, None)])
def test_steps(d, bits, dtype, kernel, mask):
    g = torch.Generator(device="cuda").manual_seed(d + bits)
    new = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=bits, residual_length=64, alpha_key=2.0, alpha_value=2.0))
    layer.update(new(3, 2, 500, d), new(3, 2, 500, d))
    reused = 0
    for step in range(600):
        layer.update(new(3, 2, 1, d), new(3, 2, 1, d), {"materialize_full_kv": False})
        if step % 7 and step % 256 > 3:  # the steps around a flush, and every seventh
            continue
        query = new(3, 4, 1, d)
        kind = ("none", "additive", "bool")[step % 3] if mask == "mixed" else mask
        m = _mask(kind, layer.get_seq_length(), dtype, g)
        call = lambda: mz.mu_zero_decode_attention_forward(_Module(), query, m, d ** -0.5, layer.get_attention_state())[0]
        cached = layer._hip_decode
        got = call()
        reused += cached is not None and layer._hip_decode is cached
        assert layer._hip_decode.kernel == kernel
        cached, layer._hip_decode = layer._hip_decode, None
        assert torch.equal(got.view(torch.int16), call().view(torch.int16)), step
        layer._hip_decode = cached
    assert reused > (20 if mask == "mixed" else 60)
