"""Dense attention over key ranges side by side (few query tiles and heads) against float64, at the edges of its rule:
the fewest key blocks, ranges of unequal length, a last block of one key, ragged query tiles, and the item counts around
256 where it stops splitting. Outputs are bf16 (half a step, 2^-8 of the value, and the probabilities' rounding to
bf16, which averages over the keys): 2e-2 and relative 1e-2 as everywhere."""
import math

import pytest
import torch

from helpers import check_close, f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lq,Lk,H", [(1, 449, 1), (128, 512, 1), (129, 513, 2), (300, 1537, 3), (1537, 1537, 12),
                                     (256, 33000, 24), (77, 40001, 1), (1280, 700, 24), (2600, 2600, 12),
                                     (2816, 575, 12), (4000, 4001, 8), (4100, 1000, 8)])
def test_split_dense_matches_float64(dev, Lq, Lk, H):
    from self_trainable_or_free_attn_amd import _lib
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    print("dense", Lq, Lk, H, "workspace", _lib.dense_workspace_bytes(Lq, Lk, H), flush=True)
    g = torch.Generator(device=dev).manual_seed(Lq + Lk)
    q = 2.0 * torch.randn(Lq, H, 128, device=dev, generator=g)
    k, v = (torch.randn(Lk, H, 128, device=dev, generator=g) for _ in range(2))
    k[Lk // 3] *= 6.0                     # one range holds far larger logits than the others
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    out, lse = K.dense_attention_kv(q, k, v) if Lq != Lk else K.dense_attention(q, k, v)
    again, lse2 = K.dense_attention_kv(q, k, v)
    assert torch.equal(out, again) and torch.equal(lse, lse2)
    assert (lse[Lq:] == 1e30).all()
    for h in range(H):
        s = q[:, h].double() @ k[:, h].double().t() / math.sqrt(128)
        ref = torch.softmax(s, -1) @ v[:, h].double()
        check_close(f"O head {h}", f32(out[:, h]), f32(ref))
        # the row sum adds the probabilities as rounded to bf16, each off by at most half a bf16 step (2^-8 of
        # itself), so the sum is too; 1e-4 for the float32 logits
        assert float((lse[:Lq, h].double() * math.log(2) - torch.logsumexp(s, -1)).abs().max()) < 2 ** -8 + 1e-4


def test_split_needs_its_workspace(dev):
    from self_trainable_or_free_attn_amd import _lib
    q = torch.randn(256, 2, 128, device=dev).bfloat16()
    k = torch.randn(2048, 2, 128, device=dev).bfloat16()
    out, lse = torch.empty_like(q), torch.empty(256, 2, device=dev)
    n = _lib.dense_workspace_bytes(256, 2048, 2)
    assert _lib.dense_workspace_bytes(1280, 512, 24) == _lib.dense_workspace_bytes(2816, 4096, 12) == 0
    assert n > 0
    for ws, size in ((None, n), (torch.empty(n - 4, device=dev, dtype=torch.uint8), n - 4)):
        with pytest.raises(RuntimeError, match="workspace|null"):
            _lib.call("es_dense_attention_ws", q, k, k, out, lse, ws, size, 256, 2048, 2, 128)


def test_split_replays_in_a_graph(dev):
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    q, k, v = (torch.randn(n, 3, 128, device=dev).bfloat16() for n in (200, 3000, 3000))
    want, wlse = K.dense_attention_kv(q, k, v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse = K.dense_attention_kv(q, k, v)
    for _ in range(3):
        out.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(lse, wlse)
        K.dense_attention_kv(q, k, v)
