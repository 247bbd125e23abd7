"""The allocation-free decode entry point (GPU).

``muzero_decode_attention_noalloc`` keeps a split call's partial records in the
library's static per-device scratch instead of a caller workspace.  Through the
C ABI it must give the workspace entry point's output bit for bit, on calls
that use the scratch (split over tokens) for the codebook, fold and general
kernels, two calls in a row (the second one smaller, so it reads only what it
wrote over the first call's records), and for a single-split call, which
needs no scratch.  The rejection of a call whose partials exceed the scratch
is host logic, checked on the CPU in test_abi.py.
"""

import ctypes

import pytest
import torch

from oracle import reference_torch as ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _plan(B, hkv, length, bits, seed, n_split=0, kernel_path="auto"):
    from muzero_amd.kernels import loader as L
    k, v, q, _ = ref.synthetic_kv(B, hkv, length, 128, hkv * 4, seed=seed)
    _, st = ref.reference_decode(q, k, v, bits=bits, alpha_k=2.0, alpha_v=2.0, group_size=64, residual=128)
    d = lambda t: t.to(DEV)
    return L.DecodePlan(d(q), bits=bits, n_groups=st["lq"] // 64, k_packed=d(st["packed_k"]), k_mn=d(st["k_mn"]),
                        k_scale=d(st["k_scale"]), v_packed=d(st["packed_v"]), v_mn=d(st["v_mn"]),
                        v_scale=d(st["v_scale"]), k_res=d(st["res_k"]), v_res=d(st["res_v"]), alpha_key=2.0,
                        alpha_value=2.0, scaling=128 ** -0.5, n_split=n_split, kernel_path=kernel_path)


def _noalloc(plan):
    """Launch the plan's arguments through muzero_decode_attention_noalloc into a fresh output
    (no workspace passed)."""
    from muzero_amd import _lib
    out = torch.full_like(plan.out, float("nan"))
    a = _lib.DecodeArgs.from_buffer_copy(plan.args)
    a.out = out.data_ptr()
    a.workspace, a.workspace_bytes = None, 0
    st = _lib.load().muzero_decode_attention_noalloc(ctypes.byref(a), _lib.stream_ptr(out.device))
    return st, out


@pytest.mark.parametrize("bits,kernel_path,kernel", [(4, "auto", "codebook"), (2, "auto", "codebook"),
                                                     (1, "auto", "codebook"), (4, "fold", "fold"), (6, "auto", "fold"),
                                                     (8, "auto", "twopass"), (8, "general", "general"),
                                                     (4, "general", "general")])
def test_noalloc_matches_workspace_entry_point(bits, kernel_path, kernel):
    """The codebook kernel (1, 2, 4 bits), the fold kernel (6 bits, and 4 bits forced onto it), the
    two-pass kernel (8 bits: its split records and logits in the scratch) and the general kernel (8 bits
    and 4 bits forced onto it), both calls split over tokens."""
    for B, hkv, length, seed in ((2, 2, 4096, 1), (1, 1, 1024, 2)):
        plan = _plan(B, hkv, length, bits, seed, kernel_path=kernel_path)
        assert plan.kernel == kernel  # the kernel this case is meant to send through the scratch
        assert plan.n_split > 1  # the call goes through the scratch
        want = plan.run().clone()
        st, got = _noalloc(plan)
        torch.cuda.synchronize()
        assert st == 0, st
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (B, hkv, length)


def test_noalloc_single_split():
    """A single-split call writes the output directly and needs no scratch."""
    plan = _plan(1, 2, 700, 4, 3, n_split=1)
    want = plan.run().clone()
    st, got = _noalloc(plan)
    torch.cuda.synchronize()
    assert st == 0 and torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("hkv,n_rep,length,bits,alpha_v", [(8, 8, 16384, 8, 4.0), (8, 4, 9000, 8, 4.0), (8, 8, 9000, 4, 2.0)])
def test_noalloc_takes_fewer_splits_where_the_librarys_count_does_not_fit(hkv, n_rep, length, bits, alpha_v):
    """The split count the library picks with a workspace may need more records than the scratch holds
    (8 heads, 256 splits, 8 bits: 8.6 MB before the logits); the call then runs with fewer."""
    from muzero_amd.kernels import loader as L
    g = torch.Generator(device="cuda").manual_seed(1)
    lq, d, qb = length // 64 * 64 - 64, 128, 8 * bits
    q = torch.randn(1, hkv * n_rep, 1, d, generator=g, device="cuda").bfloat16()

    def pack(shape):
        return (torch.randint(0, 256, (*shape, qb), generator=g, device="cuda", dtype=torch.uint8),
                -torch.rand(*shape, 1, generator=g, device="cuda").half() - 1, torch.rand(*shape, 1, generator=g, device="cuda").half() + 2)
    (kp, km, ks), (vp, vm, vs) = pack((1, hkv, lq // 64, d)), pack((1, hkv, lq, 2))
    res = torch.randn(2, 1, hkv, 64, d, generator=g, device="cuda").bfloat16()
    plan = L.DecodePlan(q, bits=bits, n_groups=lq // 64, k_packed=kp, k_mn=km, k_scale=ks, v_packed=vp, v_mn=vm, v_scale=vs,
                        k_res=res[0], v_res=res[1], alpha_key=2.0, alpha_value=alpha_v, scaling=d ** -0.5)
    want = plan.run().float()
    st, got = _noalloc(plan)
    assert st == 0
    assert (got.float() - want).abs().max().item() < 8e-3  # bf16 outputs below 1: at most an ulp apart


def _random_args(B, hkv, n_rep, length, bits):
    g = torch.Generator(device="cuda").manual_seed(B + length)
    lq, d, qb = length // 64 * 64 - 64, 128, 8 * bits
    q = torch.randn(B, hkv * n_rep, 1, d, generator=g, device="cuda").bfloat16()

    def pack(shape):
        meta = [torch.rand(*shape, 1, generator=g, device="cuda").half() for _ in range(2)]
        return (torch.randint(0, 256, (*shape, qb), generator=g, device="cuda", dtype=torch.uint8), -meta[0] - 1, meta[1] + 2)
    (kp, km, ks), (vp, vm, vs) = pack((B, hkv, lq // 64, d)), pack((B, hkv, lq, 2))
    res = torch.randn(2, B, hkv, 64, d, generator=g, device="cuda").bfloat16()
    return q, dict(bits=bits, n_groups=lq // 64, k_packed=kp, k_mn=km, k_scale=ks, v_packed=vp, v_mn=vm, v_scale=vs,
                   k_res=res[0], v_res=res[1], alpha_key=2.0, alpha_value=2.0, scaling=d ** -0.5)


@pytest.mark.parametrize("B,hkv,n_rep,length,kernel_path,n_split",
                         [(129, 8, 8, 2000, "general", 1), (257, 8, 4, 1000, "general", 1),  # one split needs no records
                          (4, 8, 4, 16000, "general", 0),   # the logits leave the two-pass kernel too few splits
                          (4, 8, 4, 12000, "auto", 31),     # two-pass with half of its 63 splits
                          (4, 8, 4, 15000, "auto", 6),      # with an eighth of its 59
                          (1, 8, 8, 16384, "auto", 64)])    # and with a quarter of its 256
def test_noalloc_reduces_splits_and_falls_back(B, hkv, n_rep, length, kernel_path, n_split):
    """8-bit calls beyond the scratch: the kernel and the split count they run with, bit for bit."""
    from muzero_amd.kernels import loader as L
    q, kw = _random_args(B, hkv, n_rep, length, 8)
    plan = L.DecodePlan(q, **kw)
    assert plan.kernel == "twopass" and plan.args.workspace_bytes > 8 << 20
    want = L.DecodePlan(q, kernel_path=kernel_path, n_split=n_split, **kw)
    assert want.kernel == ("general" if kernel_path == "general" else "twopass")
    st, got = _noalloc(plan)
    assert st == 0, st
    assert torch.equal(got.view(torch.int16), want.run().view(torch.int16))
