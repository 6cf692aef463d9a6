"""The one-workgroup kv->q inversion (NB <= 256) at its edges against numpy, through the CSR transpose and the global
top-k, and the dense lists of the coarse branch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NB", [1, 31, 32, 33, 64, 65, 128, 129, 192, 193, 255, 256, 257, 512])
@pytest.mark.parametrize("density", [0.0, 0.2, 1.0])
def test_csr_transpose_small(dev, NB, density):
    from self_trainable_or_free_attn_amd.vsa import _C, mask_to_selection
    H = 3
    g = torch.Generator(device=dev).manual_seed(NB)
    mask = torch.rand(1, H, NB, NB, device=dev, generator=g) < density
    if density == 0.2:
        mask[0, 1] = False
    sel = mask_to_selection(mask)
    out_ptr, out_idx = _C.csr_transpose(sel.q2k_ptr, sel.q2k_idx)
    assert torch.equal(out_ptr, sel.k2q_ptr)
    n = int(sel.k2q_ptr[0, -1, -1])
    assert torch.equal(out_idx[:n], sel.k2q_idx[:n])


@pytest.mark.parametrize("NB,budget", [(5, 7), (97, 1500), (400, 160000), (512, 12345), (300, 0)])
def test_global_topk_inversion(dev, NB, budget):
    from self_trainable_or_free_attn_amd.vsa import _C
    H = 2
    g = torch.Generator(device=dev).manual_seed(NB)
    scores = torch.randint(0, 50, (H, NB, NB), device=dev, generator=g).float()
    i32 = dict(device=dev, dtype=torch.int32)
    out = [torch.full((1, H, NB + 1), -1, **i32), torch.full((max(1, H * min(budget, NB * NB)),), -1, **i32)]
    out += [t.clone() for t in out]
    _C.global_topk_into(scores, budget, 0, *out)
    qp, qi, kp, ki = (t.cpu().numpy() for t in out)
    keff = min(budget, NB * NB)
    for h in range(H):
        order = np.argsort(-scores[h].cpu().numpy().ravel(), kind="stable")[:keff]
        mask = np.zeros(NB * NB, bool)
        mask[order] = True
        mask = mask.reshape(NB, NB)
        base = h * keff
        assert np.array_equal(qp[0, h], base + np.concatenate([[0], np.cumsum(mask.sum(1))]))
        assert np.array_equal(kp[0, h], base + np.concatenate([[0], np.cumsum(mask.sum(0))]))
        assert np.array_equal(qi[base:base + keff], np.nonzero(mask)[1])
        assert np.array_equal(ki[base:base + keff], np.nonzero(mask.T)[1])


@pytest.mark.parametrize("NB,BH", [(1, 1), (64, 3), (65, 2), (480, 24), (1857, 5)])
def test_dense_lists(dev, NB, BH):
    from self_trainable_or_free_attn_amd.vsa import _C
    T = -(-NB // 64)
    cnt, ptr, idx = _C.dense_lists(1, BH, NB, dev)
    assert cnt.tolist() == [min(64, NB - 64 * t) for t in range(T)]
    assert torch.equal(ptr[0].cpu(), torch.tensor([[(h * T + i) * T for i in range(T + 1)] for h in range(BH)],
                                                  dtype=torch.int32))
    assert torch.equal(idx.cpu(), torch.arange(T, dtype=torch.int32).repeat(BH * T))
