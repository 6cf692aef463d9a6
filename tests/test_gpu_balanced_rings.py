"""The queue-counter rings with launches large enough to take a slot (more than 512 items; smaller grids bind every
item to its dispatch slot and take none): short launches that wrap the ring while a long one holds a slot, calls on
two streams at once, and graph replays with uncaptured launches between them, byte for byte."""
import pytest
import torch

pytestmark = pytest.mark.gpu
H = 8


def _qkv(dev, Lq, Lk, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    return [torch.randn(n, H, 128, device=dev, generator=g).bfloat16() for n in (Lq, Lk, Lk)]


def test_short_launches_wrap_the_ring_under_a_long_one(dev):
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    long_in, short_in = _qkv(dev, 32768, 32768, 1), _qkv(dev, 8320, 200, 2)      # 2048 items; 576 with padding
    want_long, want_short = K.dense_attention(*long_in), K.dense_attention_kv(*short_in)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        got_long = K.dense_attention(*long_in)
    with torch.cuda.stream(b):
        got = [K.dense_attention_kv(*short_in) for _ in range(70)]
    torch.cuda.synchronize()
    for x, y in zip(got_long, want_long):
        assert torch.equal(x, y)
    for res in got:
        for x, y in zip(res, want_short):
            assert torch.equal(x, y)


def test_replays_with_uncaptured_launches_between(dev):
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    x = _qkv(dev, 8320, 300, 3)
    want = K.dense_attention_kv(*x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = K.dense_attention_kv(*x)
    for _ in range(3):
        got[0].zero_()
        graph.replay()
        other = K.dense_attention_kv(*x)
        torch.cuda.synchronize()
        for res in (got, other):
            for a, b in zip(res, want):
                assert torch.equal(a, b)


def test_vsa_launches_on_two_streams(dev):
    from self_trainable_or_free_attn_amd.vsa import _C, mask_to_selection
    NB, heads = 96, 12                                                          # 1152 items
    g = torch.Generator(device=dev).manual_seed(4)
    q, k, v, do = (torch.randn(1, heads, NB * 64, 128, device=dev, generator=g).bfloat16() for _ in range(4))
    cnt = torch.randint(1, 65, (NB,), device=dev, generator=g).to(torch.int32)
    u = torch.rand(1, heads, NB, NB, device=dev, generator=g)
    sel = mask_to_selection(u < torch.rand(1, heads, NB, 1, device=dev, generator=g))     # lists of every length

    def run():
        o, lse = _C.attn_fwd(q, k, v, sel.q2k_ptr, sel.q2k_idx, cnt)
        delta = _C.row_dot(do, o, cnt)
        dk, dv = _C.attn_bwd(q, k, v, do, lse, delta, sel.k2q_ptr, sel.k2q_idx, cnt)
        return o, lse, dk, dv, _C.attn_bwd_q(q, k, v, do, lse, delta, sel.q2k_ptr, sel.q2k_idx, cnt)

    want = run()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for _ in range(15):
        for s in streams:
            with torch.cuda.stream(s):
                got.append(run())
    torch.cuda.synchronize()
    for res in got:
        for a, b in zip(res, want):
            assert torch.equal(a, b)
