"""Dense K / V from packed blocks (muzero_dequantize_keys / _values) against the oracle, bit for bit:
head dims around the kernels' lane and chunk widths, every code width and output type, tails, strided
storage, short and long blocks (whole groups per lane and quarters), and non-finite metadata."""

import pytest
import torch

from muzero_amd.kernels import loader as L
from oracle import reference_torch as ref

pytestmark = pytest.mark.gpu
BF, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _packed(kind, b, h, tokens, d, bits, meta, seed):
    g = torch.Generator().manual_seed(seed)
    n, inner = (tokens // 64, d) if kind == "key" else (tokens, -(-d // 64))
    packed = torch.randint(0, 256, (b, h, n, inner, 8 * bits), generator=g, dtype=torch.uint8)
    mn = torch.randn(b, h, n, inner, 1, generator=g) * 2 - 1
    sc = torch.rand(b, h, n, inner, 1, generator=g) * 4 + 1e-3
    return packed, mn.to(meta), sc.to(meta)


def _oracle(kind, packed, mn, sc, bits, alpha, d, dtype):
    if kind == "key":
        return ref.dequantize_key_block(packed, mn, sc, bits, alpha, 64, dtype)
    return ref.dequantize_value_block(packed, mn, sc, bits, alpha, 64, d, dtype)


def _same(got, want):
    assert got.shape == want.shape and got.dtype == want.dtype
    kind = torch.int32 if got.dtype == F32 else torch.int16
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.masked_fill(nan, 0).view(kind), want.masked_fill(nan, 0).view(kind))


@pytest.mark.parametrize("kind", ["key", "value"])
@pytest.mark.parametrize("bits", range(1, 9))
@pytest.mark.parametrize("dtype,meta", [(BF, F16), (F16, BF), (F32, F32)])
@pytest.mark.parametrize("d", [33, 64, 80, 128, 200])
def test_block(kind, bits, dtype, meta, d):
    tokens = 192 if kind == "key" else 131
    packed, mn, sc = _packed(kind, 2, 3, tokens, d, bits, meta, bits * 1000 + d)
    want = _oracle(kind, packed, mn, sc, bits, 4.0, d, dtype)
    tail = torch.randn(2, 3, 150, d).to(dtype)[:, :, 3:-26]  # strided, 121 tokens
    got = L.dequantize_block(packed.cuda(), mn.cuda(), sc.cuda(), kind, bits, 4.0, d, dtype, tail.cuda()).cpu()
    _same(got[:, :, :tokens], want)
    _same(got[:, :, tokens:], tail)


@pytest.mark.parametrize("kind", ["key", "value"])
@pytest.mark.parametrize("bits,d", [(4, 128), (2, 64), (8, 128), (3, 96)])
def test_long_block_in_larger_storage(kind, bits, d):
    """Enough groups for whole groups per lane, read as views of longer capacity buffers, no tail."""
    packed, mn, sc = _packed(kind, 8, 8, 64 * 80, d, bits, F16, 5)
    n = packed.shape[2] - 5 if kind == "key" else packed.shape[2] - 64 * 5
    dev = [t.cuda()[:, :, :n] for t in (packed, mn, sc)]
    got = L.dequantize_block(*dev, kind, bits, 2.0, d, BF).cpu()
    for b in (0, 7):
        _same(got[b:b + 1], _oracle(kind, packed[b:b + 1, :, :n], mn[b:b + 1, :, :n], sc[b:b + 1, :, :n], bits, 2.0, d, BF))


@pytest.mark.parametrize("bits", [1, 4, 8])
@pytest.mark.parametrize("dtype", [BF, F16, F32])
def test_non_finite_metadata_and_misaligned_rows(bits, dtype):
    """NaN / infinite minima and scales give what the oracle's fp32 operations give; rows stored at an
    odd element offset take the element-wise stores."""
    packed, mn, sc = (t.reshape(-1, t.shape[-1]) for t in _packed("value", 1, 1, 100, 64, bits, F32, 9))
    bad = [(float("nan"), 1.0), (1.0, float("inf")), (float("-inf"), 1.0), (float("inf"), 2.0),
           (float("-inf"), float("inf")), (0.0, float("inf")), (3.0e38, 3.0e38), (-5.0, 1.0), (5.0, 1.0)]
    for i, (m, s) in enumerate(bad):
        mn[7 * i], sc[7 * i] = m, s
    want = ref.dequantize_rows(packed, mn, sc, bits, 2.0, 64, dtype)
    out = torch.empty(100 * 64 + 1, dtype=dtype, device="cuda")[1:].view(100, 64)
    L.mu_zero_dequantize_cuda(packed.cuda(), mn.cuda(), sc.cuda(), out, bits, 2.0)
    _same(out.cpu(), want)


def test_dense_read_keeps_the_tail_in_the_graph():
    """With a residual that requires grad, the dense read differentiates to its tokens."""
    import muzero_amd as mz
    layer = mz.MuZeroCacheLayer(mz.MuZeroConfig(bits=4))
    k, v = torch.randn(2, 1, 2, 300, 64, device="cuda", dtype=BF)
    layer.update(k, v)
    tail = layer.keys.clone().requires_grad_()
    layer._set_tail(tail, layer.values)
    dense, _ = layer.dense_kv()
    plain_layer_keys = torch.cat([layer._dequantize_key_prefix(), tail.detach()], 2)
    assert torch.equal(dense.detach(), plain_layer_keys)
    dense.float().sum().backward()
    assert torch.equal(tail.grad, torch.ones_like(tail))


@pytest.mark.parametrize("first,then", [((BF, BF), (F32, F32)), ((F16, F16), (BF, BF)), ((BF, F32), (BF, F32))])
def test_dense_read_promotes_a_tail_of_another_dtype(first, then):
    """A chunk in another dtype than the first, or values in another dtype than the keys: the prefix comes in the
    layer dtype (the keys' first), and the whole is promoted with the tail as concatenation promotes it."""
    import muzero_amd as mz
    g = torch.Generator(device="cuda").manual_seed(4)
    new = lambda t, dtype: torch.randn(1, 2, t, 64, generator=g, device="cuda").to(dtype)
    layer = mz.MuZeroCacheLayer(mz.MuZeroConfig(bits=4, residual_length=128))
    layer.update(new(512, first[0]), new(512, first[1]))
    got = layer.update(new(7, then[0]), new(7, then[1]))
    prefix = layer._dequantize_key_prefix(), layer._dequantize_value_prefix()
    for dense, head, tail in zip(got, prefix, (layer.keys, layer.values)):
        assert head.dtype == first[0] and head.shape[2] == 384 and tail.shape[2] == 135
        want = torch.cat([head, tail], 2)
        assert dense.dtype == want.dtype and torch.equal(dense, want)
    assert got[1].dtype == F32
