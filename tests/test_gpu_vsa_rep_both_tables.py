"""Both tiers' table gradients in one launch equal the two single-tier launches bit for bit: head counts that the eight
queues do not divide, block counts around the 64-row groups, every mid_reps."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,NB,RM", [(1, 1, 4), (3, 16, 4), (9, 17, 1), (2, 65, 2), (5, 33, 8), (8, 130, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_both_tables_equal_single_tiers(dev, BH, NB, RM, dtype):
    from self_trainable_or_free_attn_amd import _lib
    from self_trainable_or_free_attn_amd.vsa import _C
    from self_trainable_or_free_attn_amd.vsa.rep import pack_bits
    L = NB * 64
    g = torch.Generator(device=dev).manual_seed(NB)
    q, k, v, do = (torch.randn(1, BH, L, 128, device=dev, generator=g).to(dtype) for _ in range(4))
    cnt = torch.randint(1, 65, (NB,), device=dev, generator=g).to(torch.int32)
    u = torch.rand(1, BH, NB, NB, device=dev, generator=g)
    bits_a, bits_ab = pack_bits(u < 0.2), pack_bits(u < 0.5)
    tab = _C.rep_build(k, v, cnt, RM)
    lse = torch.randn(1, BH, L, device=dev, generator=g) + 5
    delta = torch.randn(1, BH, L, device=dev, generator=g)
    grads = lambda: [torch.randn(t.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(1))
                     for t in (tab[0], tab[1], tab[3], tab[4])]
    one, two = grads(), grads()
    s = "_f16" if dtype == torch.float16 else ""
    stats = (lse, delta, bits_a, bits_ab)
    _lib.call("vsa_rep_bwd_both_tables" + s, q, do, tab[0], tab[1], tab[2], 0, tab[3], tab[4], tab[5], *stats, *one, BH,
              L, 128, RM)
    _lib.call("vsa_rep_bwd_tables" + s, q, do, tab[0], tab[1], tab[2], 0, *stats, two[0], two[1], BH, L, 128, RM, 2)
    _lib.call("vsa_rep_bwd_tables" + s, q, do, tab[3], tab[4], tab[5], 0, *stats, two[2], two[3], BH, L, 128, RM, 4)
    for a, b in zip(one, two):
        assert torch.equal(a, b)
        assert torch.isfinite(a).all()
