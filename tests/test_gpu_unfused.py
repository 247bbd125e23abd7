"""The default decode path in four launches (muzero_decode_unfused) against the same path step by step
(muzero_qk, torch matmuls and softmax, muzero_av): head dims around the kernels' chunks, head counts, types,
masks, residuals shorter and longer than a workgroup's share, rows longer than the softmax holds in LDS, the
per-token value flush, and no prefix at all."""

import pytest
import torch

import muzero_amd as mz
from muzero_amd.cache import attention as A
from muzero_amd.cache.layer import MuZeroCacheLayer

pytestmark = pytest.mark.gpu
BF, F16, F32 = torch.bfloat16, torch.float16, torch.float32


class _Module:
    def __init__(self, n_rep):
        self.num_key_value_groups = n_rep


def _both(B, hkv, n_rep, d, tokens, bits, dtype, residual=128, mask=False, logq=False, meta="float16", seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + d + tokens)
    k, v = (torch.randn(B, hkv, tokens, d, generator=g, device="cuda").to(dtype) for _ in range(2))
    q = torch.randn(B, hkv * n_rep, 1, d, generator=g, device="cuda").to(dtype)
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=bits, residual_length=residual, amax_dtype=meta, alpha_key=2.0,
                                             alpha_value=2.0, logq_compatible_layout=logq))
    layer.update(k[:, :, :-1], v[:, :, :-1])
    layer.update(k[:, :, -1:], v[:, :, -1:], {"materialize_full_kv": False})
    st = layer.get_attention_state()
    m = None
    if mask:
        m = torch.zeros(B, 1, 1, tokens, dtype=dtype, device="cuda")
        m[0, ..., :tokens // 3] = torch.finfo(dtype).min
    got = mz.mu_zero_decode_attention_forward(_Module(n_rep), q, m, d ** -0.5, st)[0]
    again = mz.mu_zero_decode_attention_forward(_Module(n_rep), q.clone(), m, d ** -0.5, st)[0]  # the cached arguments
    assert torch.equal(got.view(torch.uint8), again.view(torch.uint8))
    want = A._split_steps(layer, n_rep, q, A._k.prepare_mask(m, B, tokens), d ** -0.5, st["key_prefix_length"],
                          st["value_prefix_length"], layer.keys, layer.values, 2.0, 2.0)
    return got, want


def _check(got, want):
    """Logits, weights and the output are rounded at the same places; sums in another order move a few of
    them to the neighbouring value, so the outputs lie within a few units of the type's rounding."""
    assert got.shape == want.shape and got.dtype == want.dtype
    eps = {BF: 2.0 ** -8, F16: 2.0 ** -11, F32: 2.0 ** -19}[got.dtype]
    rel = (got.double() - want.double()).norm() / want.double().norm()
    assert rel.item() < 4 * eps, rel.item()


@pytest.mark.parametrize("d", [16, 33, 80, 96, 200, 256])
@pytest.mark.parametrize("n_rep,bits,dtype", [(1, 4, BF), (3, 8, F16), (4, 2, F32), (8, 3, BF), (16, 7, BF)])
def test_shapes(d, n_rep, bits, dtype):
    _check(*_both(2, 2, n_rep, d, 777, bits, dtype, mask=n_rep == 3, meta="float32" if dtype == F32 else "bfloat16"))


@pytest.mark.parametrize("tokens,residual", [(70, 128), (300, 640), (2100, 320), (14000, 128), (12289, 64)])
def test_lengths(tokens, residual):
    _check(*_both(1, 2, 4, 96, tokens, 4, BF, residual=residual, mask=True))


@pytest.mark.parametrize("dtype", [BF, F32])
def test_values_flushed_per_token(dtype):
    _check(*_both(2, 2, 4, 96, 500, 4, dtype, residual=64, logq=True))


def test_derivatives_run_the_steps():
    """A query that requires grad keeps the step-by-step path, which differentiates through the residual."""
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=4))
    k, v = torch.randn(2, 1, 2, 100, 96, device="cuda", dtype=F32)
    layer.update(k, v)
    q = torch.randn(1, 4, 1, 96, device="cuda", requires_grad=True)
    out, _ = mz.mu_zero_decode_attention_forward(_Module(2), q, None, 0.1, layer.get_attention_state())
    out.sum().backward()
    assert q.grad is not None and torch.isfinite(q.grad).all()


def test_a_layer_holds_no_large_workspace_between_calls():
    """The workspace holds all logits of a call: only the output may stay allocated after one, on the call that
    builds the layer's arguments and on those that re-use them."""
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=4, residual_length=128))
    k, v = torch.randn(2, 4, 2, 60000, 96, device="cuda").to(BF)
    layer.update(k[:, :, :-1], v[:, :, :-1])
    layer.update(k[:, :, -1:], v[:, :, -1:], {"materialize_full_kv": False})
    q = torch.randn(4, 8, 1, 96, device="cuda").to(BF)
    logits = 4 * 8 * 60000 * 2
    torch.cuda.synchronize()
    for _ in range(3):
        before = torch.cuda.memory_allocated()
        out, _ = mz.mu_zero_decode_attention_forward(_Module(4), q, None, 0.1, layer.get_attention_state())
        assert torch.cuda.memory_allocated() - before < logits // 4


def test_a_workspace_that_outgrows_what_a_layer_keeps(monkeypatch):
    """Steps across the bound, both ways, give what new arguments give."""
    g = torch.Generator(device="cuda").manual_seed(1)
    new = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(BF)
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=4, residual_length=64))
    layer.update(new(2, 2, 300, 96), new(2, 2, 300, 96))
    kept, bounds = [], A._k.StepDecode.KEPT_WORKSPACE
    call = lambda q: mz.mu_zero_decode_attention_forward(_Module(4), q, None, 0.1, layer.get_attention_state())[0]
    for step in range(40):
        layer.update(new(2, 2, 1, 96), new(2, 2, 1, 96), {"materialize_full_kv": False})
        q = new(2, 8, 1, 96)
        if step == 2:  # between this step's workspace and that of one some tokens later
            bounds = layer._hip_decode.args.workspace_bytes + 200
        monkeypatch.setattr(A._k.StepDecode, "KEPT_WORKSPACE", bounds if step < 30 else 2 << 20)
        got = call(q)
        cached = layer._hip_decode
        kept.append(cached.workspace is not None)
        layer._hip_decode = None
        assert torch.equal(got.view(torch.int16), call(q).view(torch.int16)), step
        layer._hip_decode = cached
    assert kept[3] and not kept[29] and kept[39]


@pytest.mark.parametrize("fault", ["heads", "values"])
def test_inconsistent_calls_are_refused(fault):
    """Query heads that are not kv heads * num_key_value_groups (here of a layer without a residual, which alone would
    tell), and a value residual longer than the tokens it is said to hold."""
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=4, residual_length=0 if fault == "heads" else 64))
    k, v = torch.randn(2, 1, 2, 256, 96, device="cuda").to(BF)
    layer.update(k, v)
    state = layer.get_attention_state()
    if fault == "values":
        layer._set_tail(layer.keys[:, :, :60], layer.values)
    q = torch.randn(1, 8, 1, 96, device="cuda").to(BF)
    with pytest.raises((mz.kernels.loader.MuZeroHipError, RuntimeError)):
        mz.mu_zero_decode_attention_forward(_Module(2 if fault == "heads" else 4), q, None, 0.1, state)
