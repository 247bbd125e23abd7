"""The merged state of a packed prefix against its own records merged in 64 bits, over split counts around the
merge kernel's wave, run and lane limits (8 records a run, 64 a pass), with records that carry no weight."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _merged(acc, m, l):
    acc, m, l = acc.double(), m.double(), l.double()
    live = l > 0
    top = torch.where(live, m, -torch.inf).amax(-1)
    weight = torch.where(live, torch.exp(m - top[..., None]), 0.0)
    return (weight[..., None] * torch.where(live[..., None], acc, 0.0)).sum(-2), top, (weight * l).sum(-1)


@pytest.mark.parametrize("d,bits", [(128, 4), (64, 4), (128, 8)])
@pytest.mark.parametrize("splits", [1, 2, 8, 9, 33, 64, 65, 130])
@pytest.mark.parametrize("masked", [False, True])
def test_merged_state(d, bits, splits, masked):
    from muzero_amd.kernels import loader as L
    g = torch.Generator(device="cuda").manual_seed(splits + d)
    B, hkv, hq, qb, groups = 2, 2, 8, 8 * bits, splits

    def pack(shape):
        meta = [torch.rand(*shape, 1, generator=g, device="cuda").half() for _ in range(2)]
        return (torch.randint(0, 256, (*shape, qb), generator=g, device="cuda", dtype=torch.uint8), -meta[0] - 1, meta[1] + 2)
    (kp, km, ks), (vp, vm, vs) = pack((B, hkv, groups, d)), pack((B, hkv, 64 * groups, d // 64))
    q = 4 * torch.randn(B, hq, 1, d, generator=g, device="cuda").bfloat16()
    mask = None
    if masked:  # the first sequence's first third of the groups, and all but the last of the second's
        mask = torch.zeros(B, 1, 1, 64 * groups, device="cuda")
        mask[0, ..., :groups // 3 * 64] = float("-inf")
        mask[1, ..., :(groups - 1) * 64] = float("-inf")
    plan = L.DecodePlan(q, bits=bits, n_groups=groups, k_packed=kp, k_mn=km, k_scale=ks, v_packed=vp, v_mn=vm, v_scale=vs,
                        k_res=None, v_res=None, alpha_key=2.0, alpha_value=2.0, scaling=d ** -0.5, n_split=splits,
                        attention_mask=mask)
    new = lambda *shape: torch.full(shape, float("nan"), device="cuda")
    acc, m, l = new(B, hq, d), new(B, hq), new(B, hq)
    parts = new(B * hq, splits, d), new(B * hq, splits), new(B * hq, splits)
    plan.prefix_state(acc, m, l, *parts)
    want = _merged(*parts)
    if masked and splits > 1:
        assert (parts[2].reshape(B, hq, splits)[1, :, :-1] == 0).all()
    assert torch.equal(m.reshape(-1).double(), want[1])
    # the sums' order and __expf: a few units of fp32
    for got, exact in ((acc.reshape(B * hq, d), want[0]), (l.reshape(-1), want[2])):
        assert torch.isfinite(got).all()
        assert ((got.double() - exact).norm() / exact.norm()).item() < 2e-6
