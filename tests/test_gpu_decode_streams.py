"""One cache layer read from two streams, and from a captured graph: each call's workspace is its own."""

import pytest
import torch

import muzero_amd as mz
from muzero_amd.cache.layer import MuZeroCacheLayer

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


class _Module:
    num_key_value_groups = 4


def _layer(d, tokens, bits):
    g = torch.Generator(device="cuda").manual_seed(d + tokens + bits)
    k, v = torch.randn(2, 2, 2, tokens, d, generator=g, device="cuda").to(BF)
    layer = MuZeroCacheLayer(mz.MuZeroConfig(bits=bits, residual_length=128, alpha_key=2.0, alpha_value=2.0))
    layer.update(k[:, :, :-1], v[:, :, :-1])
    layer.update(k[:, :, -1:], v[:, :, -1:], {"materialize_full_kv": False})
    queries = torch.randn(8, 2, 8, 1, d, generator=g, device="cuda").to(BF)
    mask = torch.zeros(2, 1, 1, tokens, dtype=BF, device="cuda")
    mask[0, ..., :tokens // 3] = torch.finfo(BF).min
    return layer, queries, mask


def _call(layer, q, mask):
    return mz.mu_zero_decode_attention_forward(_Module(), q, mask, q.shape[-1] ** -0.5, layer.get_attention_state())[0]


# the fused kernels (codebook, two-pass with its logits in the workspace) and the unfused path
CASES = [(128, 4000, 4), (128, 4000, 8), (96, 3000, 4)]


@pytest.mark.parametrize("d,tokens,bits", CASES)
@pytest.mark.parametrize("masked", [False, True])
def test_two_streams(d, tokens, bits, masked):
    layer, queries, mask = _layer(d, tokens, bits)
    mask = mask if masked else None
    want = [_call(layer, q, mask).clone() for q in queries]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for _ in range(4):
        for i, q in enumerate(queries):
            with torch.cuda.stream(streams[i % 2]):
                got.append(_call(layer, q, mask))
    torch.cuda.synchronize()
    for i, out in enumerate(got):
        assert torch.equal(out.view(torch.int16), want[i % len(queries)].view(torch.int16)), i


@pytest.mark.parametrize("d,tokens,bits", CASES)
@pytest.mark.parametrize("masked", [False, True])
def test_captured_after_an_eager_call_on_the_same_stream(d, tokens, bits, masked):
    """The graph's launches write memory of the graph, whatever the layer's cached arguments become later."""
    layer, queries, mask = _layer(d, tokens, bits)
    mask = mask if masked else None
    stream = torch.cuda.Stream()
    static = queries[0].clone()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        _call(layer, static, mask)
        cached = layer._hip_decode
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = _call(layer, static, mask)
        assert layer._hip_decode is cached
        for q in queries[:4]:
            want = _call(layer, q, mask).clone()
            static.copy_(q)
            graph.replay()
            stream.synchronize()
            assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    torch.cuda.synchronize()
    del graph
