"""The queue-counter rings with launches large enough to take a slot (more than 512 items, padding included; smaller
grids bind every item to its dispatch slot and take none, but for the table gradients, which always claim): short launches
that wrap the ring while a long one holds a slot, every balanced kernel on three streams at once with more launches than
the ring has slots, and graph replays with uncaptured launches between them, byte for byte."""
import pytest
import torch

pytestmark = pytest.mark.gpu
H = 8


def _qkv(dev, Lq, Lk, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    return [torch.randn(n, H, 128, device=dev, generator=g).bfloat16() for n in (Lq, Lk, Lk)]


@pytest.mark.parametrize("short", ["dense", "sparse", "full_step"])
def test_short_launches_wrap_the_ring_under_a_long_one(dev, short):
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    print("under a long launch:", short, flush=True)
    long_in, short_in = _qkv(dev, 32768, 32768, 1), _qkv(dev, 8320, 200, 2)      # 2048 items; 576 with padding
    run = (lambda: K.dense_attention_kv(*short_in)) if short == "dense" else _launch(dev, short)
    want_long, want_short = K.dense_attention(*long_in), run()
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        got_long = K.dense_attention(*long_in)
    with torch.cuda.stream(b):
        got = [run() for _ in range(70)]
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


def _es_launches(dev):
    """The full-block step (es_block_attention) and the sparse step (es_sparse_attention) on lists of every length."""
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    L, heads = 4152, 16
    nq, nb = -(-L // 128), -(-L // 64)
    assert 8 * heads * -(-nq // 8) > 512
    g = torch.Generator(device=dev).manual_seed(7)
    q, k, v = (torch.randn(L, heads, 128, device=dev, generator=g).bfloat16() for _ in range(3))
    offset = K.dense_attention(q, k, v)[1]
    reps = K.Representatives(L, heads, 128, dev)
    km, vm = (torch.empty(nb, heads, 128, device=dev, dtype=torch.bfloat16) for _ in range(2))
    reps.build(q, k, v, km, vm)
    order = torch.rand(nq, heads, nb, device=dev, generator=g).argsort(-1).argsort(-1)
    n = torch.randint(1, nb + 1, (nq, heads, 1), device=dev, generator=g)
    r = torch.minimum(torch.randint(0, 21, (nq, heads, 1), device=dev, generator=g), nb - n)

    def lists(mask, width):
        ids = torch.where(mask, torch.arange(nb, device=dev), nb).sort(-1).values[..., :width]
        return ids.int().contiguous(), mask.sum(-1).int().contiguous()

    blocks, counts = lists(order < n, nb)
    refine, refine_counts = lists((order >= n) & (order < n + r), 32)
    means, mean_counts = lists(order >= n + r, nb)
    every, full = lists(order >= 0, nb)

    def outputs():
        return (torch.full_like(q, 7.0), torch.full((nq * 128, heads), 7.0, device=dev),
                torch.full((nq, heads), 7, device=dev, dtype=torch.int32), torch.zeros(heads, nq, nb, device=dev))

    def sparse():
        o = outputs()
        K.sparse_attention(q, k, v, km, vm, means, mean_counts, o[0], counts, blocks, offset, o[1], o[2], refine,
                           refine_counts, reps.k, reps.v, reps.log_counts, mass=o[3])
        return o

    def full_step():
        o = outputs()
        K.block_attention(q, k, v, o[0], full, every, offset, o[1], o[2], mass=o[3])
        return o

    return sparse, full_step


def _rep_launches(dev):
    """The three-tier forward, and dQ with both tables' gradients."""
    from self_trainable_or_free_attn_amd.vsa import _C, mask_to_selection
    from self_trainable_or_free_attn_amd.vsa.rep import pack_bits
    NB, heads, RM = 96, 12, 4
    assert 8 * heads * -(-NB // 8) > 512
    g = torch.Generator(device=dev).manual_seed(9)
    q, k, v, do = (torch.randn(1, heads, NB * 64, 128, device=dev, generator=g).bfloat16() for _ in range(4))
    cnt = torch.randint(1, 65, (NB,), device=dev, generator=g).to(torch.int32)
    u = torch.rand(1, heads, NB, NB, device=dev, generator=g)
    cut = 0.4 * torch.rand(1, heads, NB, 1, device=dev, generator=g)
    sel = mask_to_selection(u < cut)
    bits = pack_bits(u < cut), pack_bits(u < cut + 0.3)
    tab = _C.rep_build(k, v, cnt, RM)

    def fwd():
        return _C.rep_attn_fwd(q, k, v, *tab, sel.q2k_ptr, sel.q2k_idx, *bits, cnt, RM, 7)

    o, lse = fwd()
    delta = _C.row_dot(do, o, cnt)

    def bwd():
        grads = [torch.zeros(t.shape, device=dev) for t in (tab[0], tab[1], tab[3], tab[4])]
        dq = _C.rep_attn_bwd_q(q, k, v, *tab, do, lse, delta, sel.q2k_ptr, sel.q2k_idx, *bits, cnt, *grads, RM, 7)
        return (dq, *grads)

    return fwd, bwd


def _launch(dev, name):
    pair = {"sparse": _es_launches, "full_step": _es_launches, "rep_fwd": _rep_launches, "rep_bwd": _rep_launches}[name]
    return pair(dev)[name in ("full_step", "rep_bwd")]


@pytest.mark.parametrize("name", ["sparse", "full_step", "rep_fwd", "rep_bwd"])
def test_three_streams_wrap_the_ring(dev, name):
    print("three streams:", name, flush=True)
    run = _launch(dev, name)
    want = run()
    assert all(torch.isfinite(x).all() for x in want if x.dtype == torch.bfloat16)
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in range(3)], []
    for _ in range(25):                                                         # 75 launches of 64 slots
        for s in streams:
            with torch.cuda.stream(s):
                got.append(run())
    torch.cuda.synchronize()
    for res in got:
        for a, b in zip(res, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("name", ["sparse", "full_step", "rep_fwd", "rep_bwd"])
def test_captured_launches_replay(dev, name):
    print("replays:", name, flush=True)
    run = _launch(dev, name)
    want = run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(3):
        for x in got:
            x.fill_(3)
        graph.replay()
        other = run()
        torch.cuda.synchronize()
        for res in (got, other):
            for a, b in zip(res, want):
                assert torch.equal(a, b)
