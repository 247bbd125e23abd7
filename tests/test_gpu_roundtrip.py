"""The fused round trip (muzero_roundtrip) against quantize_rows + dequantize_rows over the same groups, bit for
bit: types, widths, head dims around its 64-channel blocks, strided inputs, constant and non-finite groups."""

import pytest
import torch
import torch.nn.functional as F

import muzero_amd as mz

pytestmark = pytest.mark.gpu


def _rows(x, kind, bits, alpha, meta):
    """The round trip through the row kernels."""
    b, h, t, d = x.shape
    if kind == "key":
        rows = x.reshape(b, h, t // 64, 64, d).transpose(3, 4).reshape(-1, 64)
    else:
        rows = F.pad(x, (0, -d % 64)).reshape(-1, 64)
    q = mz.quantize_rows(rows.float(), bits, alpha, 1e-8, meta)
    y = mz.dequantize_rows(*q, bits, alpha, 64, x.dtype)
    if kind == "key":
        return y.reshape(b, h, t // 64, d, 64).transpose(3, 4).reshape(b, h, t, d)
    return y.reshape(b, h, t, -1)[..., :d]


def _same(a, b):
    nan = torch.isnan(b)
    assert a.shape == b.shape and torch.equal(torch.isnan(a), nan)
    kind = torch.int32 if a.element_size() == 4 else torch.int16
    assert torch.equal(a.masked_fill(nan, 0).contiguous().view(kind), b.masked_fill(nan, 0).contiguous().view(kind))


@pytest.mark.parametrize("bits", range(1, 9))
@pytest.mark.parametrize("dtype,meta", [(torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16),
                                        (torch.float32, torch.float32)])
@pytest.mark.parametrize("d", [33, 64, 72, 128, 200])
def test_roundtrip(bits, dtype, meta, d):
    g = torch.Generator().manual_seed(bits + d)
    k, v = (torch.randn(2, 3, 200, d, generator=g) * 3 for _ in range(2))
    k[..., :2] *= 10
    k, v = (x.to(dtype).cuda()[:, :, 4:196] for x in (k, v))  # strided; 192 tokens
    v = v[:, :, 5:]
    rk, rv = mz.roundtrip(k, v, bits=bits, alpha_key=4.0, alpha_value=2.0, amax_dtype=meta)
    _same(rk, _rows(k, "key", bits, 4.0, meta))
    _same(rv, _rows(v, "value", bits, 2.0, meta))


@pytest.mark.parametrize("bits", [1, 4, 8])
def test_special_groups(bits):
    g = torch.Generator().manual_seed(bits)
    x = torch.randn(1, 2, 128, 128, generator=g)
    x[0, 0, :64, 3], x[0, 1, 70, :64] = 0.0, 2.5            # constant groups
    x[0, 0, 5, 7], x[0, 0, 9, 70] = float("nan"), float("inf")
    x[0, 1, 100, 100] = 3e38
    for dtype in (torch.float32, torch.bfloat16):
        y = x.to(dtype).cuda()
        rk, rv = mz.roundtrip(y, y, bits=bits, alpha_key=2.0, alpha_value=2.0)
        _same(rk, _rows(y, "key", bits, 2.0, torch.float16))
        _same(rv, _rows(y, "value", bits, 2.0, torch.float16))
