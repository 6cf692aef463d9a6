"""Backwards whose output has no gradient of its own (a loss on the log-sum-exp alone, or a later function that returns
none for it): zero gradients of the right shapes, as for a gradient of zeros, in each of the four functions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.fixture(scope="module")
def inputs(dev):
    g = torch.Generator(device=dev).manual_seed(2)
    NB, H = 7, 2
    mask = torch.rand(1, H, NB, NB, device=dev, generator=g) < 0.5
    return {D: [torch.randn(1, H, NB * 64, D, device=dev, generator=g).bfloat16() for _ in range(4)]
            for D in (64, 128)}, torch.randint(1, 65, (NB,), device=dev, generator=g).to(torch.int32), mask


def _outputs(name, q, k, v, gate, cnt, mask):
    from self_trainable_or_free_attn_amd.vsa import fine_block_sparse_attention, mask_to_selection, vsa2_attention, \
        vsa_attention
    from self_trainable_or_free_attn_amd.vsa.rep import RepTiers, rep_attention, rep_fine_attention, route_tiers
    tiers = RepTiers(frac_full=0.2, frac_mid=0.3, mid_reps=4)
    if name == "vsa":
        return vsa_attention(q, k, v, cnt, 3, weight=gate)
    if name == "vsa2":
        return vsa2_attention(q, k, v, gate, cnt, topk=3)
    if name == "rep":
        return rep_attention(q, k, v, gate, cnt, R=16, tiers=tiers)
    if name == "rep_fine":
        return rep_fine_attention(q, k, v, cnt, route_tiers(q.detach(), k.detach(), cnt, tiers), mid_reps=4)[0]
    o, lse = fine_block_sparse_attention(q, k, v, cnt, mask_to_selection(mask))
    return lse if name == "fine_lse" else o


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("name", ["vsa", "vsa2", "fine", "fine_lse", "rep", "rep_fine"])
def test_missing_output_gradient_gives_zeros(inputs, name, D):
    print("missing gradient", name, D, flush=True)
    tokens, cnt, mask = inputs
    leaves = [t.clone().requires_grad_(True) for t in tokens[D]]
    out = _outputs(name, *leaves, cnt, mask)
    if name != "fine_lse":
        out = _NoGradient.apply(out)
    used = leaves if name in ("vsa", "vsa2", "rep") else leaves[:3]
    for x, dx in zip(used, torch.autograd.grad(out.masked_fill(out == float("-inf"), 0).sum(), used)):
        assert dx.shape == x.shape and dx.dtype == x.dtype and not dx.any()
