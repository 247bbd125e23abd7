"""When a decode step may re-use the arguments cached on its layer (host logic; the launches are stand-ins that
record what reaches them, and the tensors are on the CPU)."""

import copy
import ctypes
import threading
from types import SimpleNamespace

import pytest
import torch

from muzero_amd import MuZeroConfig, mu_zero_decode_attention_forward
from muzero_amd.cache import attention as A
from muzero_amd.cache.layer import MuZeroCacheLayer

B, HKV, N_REP, D, TOKENS = 2, 2, 2, 64, 5


class _Module:
    num_key_value_groups = N_REP


class _Refused(Exception):
    """A new plan's own checks refused the call."""


class _Plan:
    """In DecodePlan's place: refuses tensors on another device, as DecodePlan does."""

    kernel = "general"

    def __init__(self, query, *, attention_mask=None, k_res=None, v_res=None, **_):
        for t in (query, attention_mask):
            if t is not None and t.device != k_res.device:
                raise _Refused
        if v_res.shape[2] != k_res.shape[2]:
            raise _Refused
        self.launches = ["plan"]

    def run(self):
        return self.launches


class _Step:
    """In StepDecode's place."""

    kernel = "general"

    def __init__(self, plan, key, stream):
        self.key, self.launches = key, plan.launches

    def launch(self, query, n_groups, n_residual, mask=None):
        self.launches.append("step")
        return self.launches


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr(A._k, "DecodePlan", _Plan)
    monkeypatch.setattr(A._k, "StepDecode", _Step)
    monkeypatch.setattr(A, "_step_owner", lambda query: (query.device, 0, 0))
    layer = MuZeroCacheLayer(MuZeroConfig(bits=4, residual_length=128))
    k, v = torch.randn(2, B, HKV, TOKENS, D).bfloat16()
    layer.update(k[:, :, :-1], v[:, :, :-1])
    layer.update(k[:, :, -1:], v[:, :, -1:], {"materialize_full_kv": False})
    return layer


def _call(layer, mask=None, device="cpu"):
    query = torch.zeros(B, HKV * N_REP, 1, D, dtype=torch.bfloat16, device=device)
    return mu_zero_decode_attention_forward(_Module(), query, mask, 0.125, layer.get_attention_state())[0]


def _mask(device="cpu"):
    return torch.zeros(B, 1, 1, TOKENS, dtype=torch.bfloat16, device=device)


def test_a_second_call_takes_the_cached_arguments(layer):
    assert list(_call(layer, _mask())) == ["plan"]
    assert list(_call(layer, _mask())) == ["plan", "step"]
    assert list(_call(layer)) == ["plan"]  # without a mask: other arguments


def test_a_mask_on_another_device_is_checked(layer):
    _call(layer, _mask())
    with pytest.raises(_Refused):
        _call(layer, _mask("meta"))
    assert list(_call(layer, _mask())) == ["plan", "step"]  # the cached arguments were not touched


def test_a_query_on_another_device_is_checked(layer):
    _call(layer)
    with pytest.raises(_Refused):
        _call(layer, device="meta")


def test_windows_of_different_lengths_are_checked(layer):
    _call(layer)
    layer._vres.end -= 1
    layer._vres._refresh()
    layer._sync()
    with pytest.raises(_Refused):
        _call(layer)


def test_other_streams_and_threads_get_their_own_arguments(layer, monkeypatch):
    """The cached arguments hold one workspace and are patched in place: another stream's launches would overwrite
    records still being read, another thread's patches the arguments of a launch under way."""
    for mask in (None, _mask()):
        for owner in ((0, 0), (1, 0), (1, 1), (0, 0)):
            monkeypatch.setattr(A, "_step_owner", lambda query, owner=owner: (query.device, *owner))
            assert list(_call(layer, mask)) == ["plan"]
            assert list(_call(layer, mask)) == ["plan", "step"]


def test_a_captured_call_neither_takes_nor_replaces_the_cached_arguments(layer, monkeypatch):
    """A graph must own the memory its launches write."""
    _call(layer)
    cached = layer._hip_decode
    monkeypatch.setattr(A, "_step_owner", lambda query: None)
    assert list(_call(layer)) == ["plan"]
    assert layer._hip_decode is cached


def test_the_owner_is_the_device_the_stream_and_the_thread(monkeypatch):
    gpu = SimpleNamespace(is_cuda=True, device=torch.device("cuda", 1))
    stream, capturing = [100], [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(A._k, "stream_ptr", lambda device: stream[0])
    assert A._step_owner(gpu) == (gpu.device, 100, threading.get_ident())
    assert A._step_owner(SimpleNamespace(is_cuda=False, device=torch.device("cpu"))) is None
    capturing[0] = True
    assert A._step_owner(gpu) is None
    stream[0], capturing[0] = 0, False
    assert A._step_owner(gpu) == (gpu.device, 0, threading.get_ident())


def test_a_copy_of_the_layer_builds_its_own_arguments(layer):
    """A cache is copied to re-use a prompt, after masked decode steps as well; the launch arguments hold addresses
    of the original's storage and cannot be copied."""
    _call(layer, _mask())
    layer._hip_decode.args = (ctypes.c_void_p * 1)(1)
    other = copy.deepcopy(layer)
    assert other._hip_decode is None and layer._hip_decode is not None
    assert torch.equal(other.keys, layer.keys) and other.keys.data_ptr() != layer.keys.data_ptr()
    assert list(_call(other, _mask())) == ["plan"]
    assert list(_call(layer, _mask())) == ["plan", "step"]
