"""The library's own split counts and the merge of many splits: every count gives the one-split result
within the kernel's rounding, and stays within the workgroups the device holds at once."""

import pytest
import torch

from muzero_amd.kernels import loader as L

pytestmark = pytest.mark.gpu


def _plan(B, hkv, n_rep, d, ctx, bits, n_split, seed=3, alpha_value=2.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    k, v = (torch.randn(B, hkv, ctx, d, generator=g, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(B, hkv * n_rep, 1, d, generator=g, device="cuda").bfloat16()
    lq, qb, ng = (ctx - 100) // 64 * 64, 8 * bits, d // 64
    packed = {}
    for name, x, shape, into in (("k", k, (B, hkv, lq // 64, d), L.quantize_key_block_into),
                                 ("v", v, (B, hkv, lq, ng), L.quantize_value_block_into)):
        pq = torch.empty((*shape, qb), dtype=torch.uint8, device="cuda")
        mn, sc = (torch.empty((*shape, 1), dtype=torch.float16, device="cuda") for _ in range(2))
        into(x[:, :, :lq], bits, 2.0 if name == "k" else alpha_value, 1e-8, pq, mn, sc)
        packed.update({f"{name}_packed": pq, f"{name}_mn": mn, f"{name}_scale": sc, f"{name}_res": x[:, :, lq:].contiguous()})
    return L.DecodePlan(q, bits=bits, n_groups=lq // 64, alpha_key=2.0, alpha_value=alpha_value, scaling=d ** -0.5,
                        n_split=n_split, out_dtype=torch.float32, **packed)


def _bound(plan, tokens):
    """How far two split counts of one call may lie apart.  A weight's own rounding (2^-17 as a high + low
    pair, 2^-11 as one fp16 in the general kernel) moves a sum of `tokens` unit values with equal weights by
    about eps / sqrt(tokens): eight times that, and 2e-6 for the fp32 sums.  The fold kernel's operands
    carry a running power-of-two scale that depends on the split: its arithmetic is held to 4e-4."""
    if plan.kernel == "fold":
        return 4e-4
    return 2e-6 + 8 * (2.0 ** -11 if plan.kernel == "general" else 2.0 ** -17) / tokens ** 0.5


@pytest.mark.parametrize("d,bits", [(128, 4), (64, 4), (128, 8), (64, 8)])
@pytest.mark.parametrize("n_split", [2, 8, 9, 17, 64, 65, 130])
def test_merge_of_many_splits(d, bits, n_split):
    """Both merge kernels (one wave up to 8 records, four above) and more records than a wave's lanes."""
    one = _plan(1, 2, 4, d, 9000, bits, 1)
    many = _plan(1, 2, 4, d, 9000, bits, n_split)
    assert (one.run() - many.run()).abs().max().item() < _bound(one, 9000)


@pytest.mark.parametrize("B,hkv,n_rep,d,ctx,bits", [
    (1, 1, 4, 128, 300, 4), (1, 8, 4, 128, 1000, 4), (3, 4, 7, 128, 2777, 3), (33, 8, 2, 128, 700, 2), (65, 8, 1, 128, 500, 4),
    (24, 8, 4, 64, 1500, 4), (2, 8, 4, 128, 3000, 7), (2, 8, 8, 128, 3000, 7), (2, 8, 4, 128, 3000, 8), (2, 8, 4, 64, 3000, 8)])
def test_own_split_count(B, hkv, n_rep, d, ctx, bits):
    own = _plan(B, hkv, n_rep, d, ctx, bits, 0)
    per_wave = own.kernel == "twopass"  # one wave per split there, one workgroup elsewhere
    slots = torch.cuda.get_device_properties(0).multi_processor_count * (8 if per_wave else 2)
    assert own.n_split == 1 or B * hkv * own.n_split <= max(slots, 2 * B * hkv)
    one = _plan(B, hkv, n_rep, d, ctx, bits, 1)
    assert own.kernel == one.kernel
    assert (own.run() - one.run()).abs().max().item() < _bound(one, ctx)
