"""Dense attention over key ranges side by side (few query tiles and heads) against float64, at the edges of its rule,
each size with the number of ranges it takes: the fewest key blocks that split (12 in three ranges, 16 in two), ranges
of unequal length, a last block of one key, ragged query tiles, the item counts around 256 where it stops splitting, and
sizes on both sides of where the merge costs more than it saves. Outputs are bf16 (half a step, 2^-8 of the value, and
the probabilities' rounding to bf16, which averages over the keys): 2e-2 and relative 1e-2 as everywhere."""
import math

import pytest
import torch

from helpers import check_close, f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lq,Lk,H,ranges", [(1, 449, 1, 1), (128, 512, 1, 1), (129, 513, 2, 1), (100, 705, 2, 3),
                                            (128, 768, 1, 3), (129, 769, 1, 3), (60, 1000, 3, 4), (1400, 960, 20, 1),
                                            (1400, 961, 20, 2), (300, 1537, 3, 6), (1537, 1537, 12, 3),
                                            (256, 33000, 24, 10), (77, 40001, 1, 16), (1280, 700, 24, 1),
                                            (2600, 2600, 12, 2), (2816, 575, 12, 1), (4000, 4001, 8, 2),
                                            (4100, 1000, 8, 1), (640, 705, 20, 1), (640, 1280, 20, 5),
                                            (2048, 1025, 12, 1), (2048, 4097, 12, 2)])
def test_split_dense_matches_float64(dev, Lq, Lk, H, ranges):
    from self_trainable_or_free_attn_amd import _lib
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    print("dense", Lq, Lk, H, "ranges", ranges, flush=True)
    partial = (128 * 128 + 2 * 128) * 4   # a range's float32 O, maximum and row sum of one 128-row query tile
    assert _lib.dense_workspace_bytes(Lq, Lk, H) == (ranges > 1) * ranges * -(-Lq // 128) * H * partial
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


def test_split_and_unsplit_calls_compile(dev):
    """Traced into one graph, with fake tensors through the Meta kernels: the eager bytes."""
    from self_trainable_or_free_attn_amd.attention import dense_attention
    for Lq, Lk in ((300, 3000), (1537, 1537), (5000, 200)):
        print("compiled dense", Lq, Lk, flush=True)
        qkv = [torch.randn(1, n, 3, 128, device=dev).bfloat16() for n in (Lq, Lk, Lk)]
        want = dense_attention(*qkv, return_lse=True)
        torch._dynamo.reset()
        f = torch.compile(lambda q, k, v: dense_attention(q, k, v, return_lse=True), backend="aot_eager", fullgraph=True)
        got = f(*qkv)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
