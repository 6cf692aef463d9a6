"""The per-row block selection at the edges of its register layouts (2, 4, 8, 16, 32 chunks of 64 columns) and of its
strip rule (8 or 32 rows per workgroup; 8 with given scores), bit for bit against the oracle. Pooled rows hold small
integers, so every dot product is exact, scores tie often and the order of ties is tested too."""
import numpy as np
import pytest
import torch

from oracle import vsa_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NB,heads,K", [(1, 2, 1), (63, 2, 5), (64, 2, 64), (65, 2, 16), (128, 3, 0), (129, 2, 40),
                                        (256, 2, 17), (257, 2, 100), (512, 1, 60), (513, 1, 60), (1024, 1, 200),
                                        (1025, 1, 1), (2048, 1, 333),
                                        (33, 1025, 7), (130, 411, 20), (200, 300, 50), (300, 205, 31), (600, 108, 40),
                                        (64, 150, 9), (64, 151, 9), (1024, 12, 9), (1024, 13, 9), (1025, 15, 9),
                                        (1025, 17, 9), (1280, 12, 30), (1281, 12, 30), (2048, 32, 17)])
@pytest.mark.parametrize("given", [False, True])
def test_row_selection_widths(dev, NB, heads, K, given):
    from self_trainable_or_free_attn_amd.vsa import _C
    print("rows", NB, heads, K, given, flush=True)
    g = torch.Generator().manual_seed(NB * 7 + heads)
    pad = (NB + 63) // 64 * 64
    qc, kc = (torch.zeros(1, heads, pad, 128) for _ in range(2))
    for x in (qc, kc):
        x[:, :, :NB, :16] = torch.randint(-2, 3, (1, heads, NB, 16), generator=g).float()
    qd, kd = qc.bfloat16().to(dev), kc.bfloat16().to(dev)
    if given:
        scores = _C.block_scores(qd, kd, NB)
        i32 = dict(device=dev, dtype=torch.int32)
        out = [torch.full((1, heads, NB + 1), -1, **i32), torch.full((heads * NB * K,), -1, **i32)]
        out += [torch.full((1, heads, NB + 1), -1, **i32), torch.full((heads * NB * K,), -1, **i32)]
        _C.row_topk_into(scores, K, 0, *out)
    else:
        out = _C.route_rows(qd, kd, NB, K)
    qp, qi, kp, ki = (x.cpu().numpy() for x in out)
    for h in sorted({0, heads // 2, heads - 1}):
        s = ref.block_scores(qc[:, h:h + 1, :NB].numpy(), kc[:, h:h + 1, :NB].numpy())
        mask = ref.row_topk_mask(s, K).reshape(NB, NB)
        base = h * NB * K
        assert np.array_equal(qp[0, h], base + np.arange(NB + 1) * K)
        assert np.array_equal(qi[base:base + NB * K], np.nonzero(mask)[1])
        assert np.array_equal(kp[0, h], base + np.concatenate([[0], np.cumsum(mask.sum(0))]))
        assert np.array_equal(ki[base:base + NB * K], np.nonzero(mask.T)[1])


@pytest.mark.parametrize("NB,heads", [(1, 1), (40, 51), (40, 52), (64, 32), (64, 33), (250, 9), (1000, 2), (1000, 3),
                                      (2048, 1), (2048, 2), (2049, 1)])
def test_block_scores_on_both_sides_of_their_strip_rule(dev, NB, heads):
    """Scores alone: 8 rows per workgroup while a launch has at most 256 workgroups, else 32."""
    from self_trainable_or_free_attn_amd.vsa import _C
    print("scores", NB, heads, flush=True)
    g = torch.Generator().manual_seed(NB + heads)
    pad = (NB + 63) // 64 * 64
    qc, kc = (torch.zeros(1, heads, pad, 128) for _ in range(2))
    for x in (qc, kc):
        x[:, :, :NB, :16] = torch.randint(-2, 3, (1, heads, NB, 16), generator=g).float()
    got = _C.block_scores(qc.bfloat16().to(dev), kc.bfloat16().to(dev), NB).float().cpu().numpy()
    for h in sorted({0, heads // 2, heads - 1}):
        want = ref.block_scores(qc[:, h:h + 1, :NB].numpy(), kc[:, h:h + 1, :NB].numpy())
        assert np.array_equal(got[h], np.asarray(want, dtype=np.float32).reshape(NB, NB))


@pytest.mark.parametrize("NB,heads", [(64, 200), (64, 201), (600, 21), (600, 22), (833, 19), (833, 20), (1000, 16),
                                      (1000, 27), (1000, 28), (1024, 32), (1025, 16)])
def test_row_selection_of_64_column_rows(dev, NB, heads):
    """Rows of 64 columns have strip lines of their own."""
    from self_trainable_or_free_attn_amd.vsa import _C
    K = 11
    print("rows of 64 columns", NB, heads, flush=True)
    g = torch.Generator().manual_seed(NB + 3 * heads)
    pad = (NB + 63) // 64 * 64
    qc, kc = (torch.zeros(1, heads, pad, 64) for _ in range(2))
    for x in (qc, kc):
        x[:, :, :NB, :16] = torch.randint(-2, 3, (1, heads, NB, 16), generator=g).float()
    qp, qi, kp, ki = (x.cpu().numpy() for x in _C.route_rows(qc.bfloat16().to(dev), kc.bfloat16().to(dev), NB, K))
    for h in sorted({0, heads // 2, heads - 1}):
        s = ref.block_scores(qc[:, h:h + 1, :NB].numpy(), kc[:, h:h + 1, :NB].numpy())
        mask = ref.row_topk_mask(s, K).reshape(NB, NB)
        base = h * NB * K
        assert np.array_equal(qp[0, h], base + np.arange(NB + 1) * K)
        assert np.array_equal(qi[base:base + NB * K], np.nonzero(mask)[1])
        assert np.array_equal(kp[0, h], base + np.concatenate([[0], np.cumsum(mask.sum(0))]))
        assert np.array_equal(ki[base:base + NB * K], np.nonzero(mask.T)[1])
