"""D = 64 rows stored 64 columns wide (VSA_PACKED_ROWS) against the same rows zero-padded to 128 columns, bit for bit,
through every entry point that takes both; and D = 64 operator calls on tensors that are not contiguous or not 16-byte
aligned, which are taken as before."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
PACKED = 64 | 0x10000


@pytest.fixture(scope="module")
def case(dev):
    B, H, NB = 1, 3, 37
    g = torch.Generator(device=dev).manual_seed(8)
    x = {n: torch.randn(B, H, NB * 64, 64, device=dev, generator=g).bfloat16() for n in ("q", "k", "v", "do", "gate")}
    cnt = torch.randint(1, 65, (NB,), device=dev, generator=g).to(torch.int32)
    from self_trainable_or_free_attn_amd.vsa import mask_to_selection
    mask = torch.rand(B, H, NB, NB, device=dev, generator=g) < 0.3
    mask[:, :, 5] = False
    return dict(x=x, cnt=cnt, sel=mask_to_selection(mask), BH=B * H, L=NB * 64, NB=NB)


def both(run):
    """run(D, widen, rows) with rows of 64 and of 128 columns; their outputs must agree on the first 64 columns and the
    wide ones be zero past them."""
    dev = "cuda"
    packed = run(PACKED, lambda t: t, lambda *s, dtype: torch.full((*s, 64), 7.0, device=dev, dtype=dtype))
    wide = run(64, lambda t: F.pad(t, (0, 64)), lambda *s, dtype: torch.full((*s, 128), 7.0, device=dev, dtype=dtype))
    for p, w in zip(packed, wide):
        if w.shape[-1] == 128 and p.shape[-1] == 64:
            assert not w[..., 64:].any()
            w = w[..., :64]
        assert torch.equal(p, w)


def test_packed_rows_equal_padded_rows(case):
    from self_trainable_or_free_attn_amd import _lib
    from self_trainable_or_free_attn_amd.vsa import _C
    c, x, cnt, sel = case, case["x"], case["cnt"], case["sel"]
    BH, L, NB = c["BH"], c["L"], c["NB"]
    bf, f32 = torch.bfloat16, torch.float32
    stat = lambda *s: torch.full(s, 3.0, device="cuda")

    def pool(D, w, rows):
        out = [rows(BH, r, dtype=bf) for r in (192, 192, 64, 64, 64)]     # 37 blocks of 4 groups, padded to 192
        _lib.call("vsa_pool", w(x["q"]), w(x["k"]), w(x["v"]), cnt, out[0], out[1], None, *out[2:], BH, L, D, 16)
        return out

    both(pool)
    qr, kr, qc, kc, oc = pool(PACKED, lambda t: t, lambda *s, dtype: torch.empty(*s, 64, device="cuda", dtype=dtype))

    def routers(D, w, rows):
        s1 = torch.zeros(BH, NB, NB, device="cuda", dtype=bf)
        _lib.call("vsa_block_scores", w(qc), w(kc), s1, NB, 64, 0, BH, D)
        lse2, s2 = stat(BH, 192), torch.zeros(BH, NB, NB, device="cuda")
        _lib.call("vsa_router_lse", w(qr), w(kr), cnt, lse2, NB, 16, BH, D)
        _lib.call("vsa_router_scores", w(qr), w(kr), lse2, cnt, s2, NB, 16, 1, 0, BH, D)
        return s1, lse2, s2

    both(routers)

    def fine(D, w, rows):
        q, k, v, do, gate = (w(x[n]) for n in ("q", "k", "v", "do", "gate"))
        o, lse = rows(BH, L, dtype=bf), stat(BH, L)
        _lib.call("vsa_attn_fwd", q, k, v, sel.q2k_ptr, sel.q2k_idx, cnt, o, lse, BH, L, D)
        fused = rows(BH, L, dtype=bf)
        _lib.call("vsa_fuse_fwd", o, w(oc), gate, fused, cnt, BH, L, D, 64, 2, 0)
        delta, dof, doc, dc, dg = stat(BH, L), rows(BH, L, dtype=bf), rows(BH, 64, dtype=bf), stat(BH, 64), \
            rows(BH, L, dtype=bf)
        _lib.call("vsa_fuse_bwd", do, o, w(oc), gate, dof, delta, doc, dc, dg, cnt, BH, L, D, 64, 2, 0)
        dot = stat(BH, L)
        _lib.call("vsa_row_dot", do, o, cnt, dot, BH, L, D)
        assert torch.allclose(dot, delta, rtol=0, atol=1e-4)     # 64 products of about 1 in float32, two orders
        out = [o, lse, fused, delta, dof, doc, dc, dg, dot]
        add = w(torch.linspace(-1, 1, BH * 64 * 64, device="cuda").view(BH, 64, 64))
        for dt, flag in ((bf, 0), (f32, 1)):
            dk, dv = rows(BH, L, dtype=dt), rows(BH, L, dtype=dt)
            _lib.call("vsa_attn_bwd_kv", q, k, v, do, lse, delta, sel.k2q_ptr, sel.k2q_idx, cnt, add, add, 64, dk, dv,
                      flag, BH, L, D)
            out += [dk, dv]
        dq, acc = rows(BH, L, dtype=bf), w(torch.ones(BH, L, 64, device="cuda"))
        _lib.call("vsa_attn_bwd_q", q, k, v, do, lse, delta, sel.q2k_ptr, sel.q2k_idx, cnt, add, 64, dq, None, BH, L, D)
        _lib.call("vsa_attn_bwd_q", q, k, v, do, lse, delta, sel.q2k_ptr, sel.q2k_idx, cnt, None, 0, None, acc, BH, L,
                  D)
        fin = rows(BH, L, dtype=bf)
        _lib.call("vsa_finalize", acc, add, 64, fin, cnt, BH, L, D)
        # split-KV: chunks of 3 blocks
        tasks, merges, info = _C.split_plan(sel.q2k_ptr, 3, 1000)
        po, pl, so, sl = rows(1000, 64, dtype=f32), stat(1000, 64), rows(BH, L, dtype=bf), stat(BH, L)
        _lib.call("vsa_attn_fwd_tasks", q, k, v, sel.q2k_idx, cnt, tasks, info, tasks.shape[0], so, sl, po, pl, BH, L,
                  D)
        _lib.call("vsa_split_merge_fwd", po, pl, merges, info, merges.shape[0], cnt, so, sl, BH, L, D, 1)
        pq, sq, sq32 = rows(1000, 64, dtype=f32), rows(BH, L, dtype=bf), w(torch.zeros(BH, L, 64, device="cuda"))
        _lib.call("vsa_attn_bwd_q_tasks", q, k, v, do, lse, delta, sel.q2k_idx, cnt, tasks, info, tasks.shape[0], add,
                  64, sq, pq, BH, L, D)
        _lib.call("vsa_split_merge_sum", pq, merges, info, merges.shape[0], add, 64, cnt, sq, None, BH, L, D)
        _lib.call("vsa_split_merge_sum", pq, merges, info, merges.shape[0], add, 64, cnt, None, sq32, BH, L, D)
        tasks, merges, info = _C.split_plan(sel.k2q_ptr, 3, 1000)
        pk, pv, sk, sv = (rows(1000, 64, dtype=f32) for _ in range(2)), None, None, None
        pk, pv = pk
        sk, sv = rows(BH, L, dtype=bf), rows(BH, L, dtype=bf)
        _lib.call("vsa_attn_bwd_kv_tasks", q, k, v, do, lse, delta, sel.k2q_idx, cnt, tasks, info, tasks.shape[0], add,
                  add, 64, sk, sv, pk, pv, BH, L, D)
        for part, dst in ((pk, sk), (pv, sv)):
            _lib.call("vsa_split_merge_sum", part, merges, info, merges.shape[0], add, 64, cnt, dst, None, BH, L, D)
        return out + [dq, acc, fin, so, sl, sq, sq32, sk, sv]

    both(fine)


def test_wrong_head_dims_stay_refused(case):
    from self_trainable_or_free_attn_amd import _lib
    c, x = case, case["x"]
    o, lse = torch.empty_like(x["q"]), torch.empty(c["BH"], c["L"], device="cuda")
    for D in (0, 32, 96, 32 | 0x10000, 64 | 0x20000, 64 | 0x30000, -64):
        with pytest.raises(RuntimeError, match="head dim must be 64 or 128"):
            _lib.call("vsa_attn_fwd", x["q"], x["k"], x["v"], c["sel"].q2k_ptr, c["sel"].q2k_idx, c["cnt"], o, lse,
                      c["BH"], c["L"], D)
    with pytest.raises(RuntimeError):
        _lib.call("vsa_row_dot", x["q"], x["k"], c["cnt"], lse, c["BH"], c["L"], 32 | 0x10000)


def test_unaligned_and_strided_d64_arguments(case):
    from self_trainable_or_free_attn_amd.vsa import _C
    c, x, cnt, sel = case, case["x"], case["cnt"], case["sel"]
    n = x["q"].numel()

    def shifted(t):   # contiguous, one element past a 16-byte boundary
        buf = torch.empty(n + 1, device="cuda", dtype=t.dtype)
        buf[1:].copy_(t.flatten())
        return buf[1:].view(t.shape)

    q, k, v = (shifted(x[i]) for i in "qkv")
    strided = lambda t: torch.cat([t, t], -1)[..., :64]
    o, lse = _C.attn_fwd(q, k, v, sel.q2k_ptr, sel.q2k_idx, cnt)
    o2, lse2 = _C.attn_fwd(x["q"], x["k"], x["v"], sel.q2k_ptr, sel.q2k_idx, cnt)
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    delta = (o.float() * x["do"].float()).sum(-1)
    args = (lse, delta, sel.k2q_ptr, sel.k2q_idx, cnt)
    for a, b in zip(_C.attn_bwd(q, k, v, strided(x["do"]), *args), _C.attn_bwd(x["q"], x["k"], x["v"], x["do"], *args)):
        assert torch.equal(a, b)
    acc = torch.zeros(1, 3, c["L"], 128, device="cuda")[..., :64]
    with pytest.raises(RuntimeError):     # (an accumulator must be contiguous, as before)
        _C.attn_bwd_q_acc(q, k, v, x["do"], lse, delta, sel.q2k_ptr, sel.q2k_idx, cnt, acc)


@pytest.mark.parametrize("D", [64, 128])
def test_compiled_fine_attention_trains_as_eager(case, D):
    from self_trainable_or_free_attn_amd.vsa import Selection, fine_block_sparse_attention
    c, sel = case, case["sel"]
    x = {n: F.pad(t, (0, D - 64)) for n, t in c["x"].items()}
    qkv = [x[n].clone().requires_grad_(True) for n in "qkv"]
    lists = (sel.q2k_ptr, sel.q2k_idx, sel.k2q_ptr, sel.k2q_idx)

    def f(q, k, v, cnt, *lists):
        return fine_block_sparse_attention(q, k, v, cnt, Selection(*lists))

    want = f(*qkv, c["cnt"], *lists)
    grads = torch.autograd.grad(want[0], qkv, x["do"])
    torch._dynamo.reset()
    got = torch.compile(f, backend="aot_eager", fullgraph=True)(*qkv, c["cnt"], *lists)
    for a, b in zip((*got, *torch.autograd.grad(got[0], qkv, x["do"])), (*want, *grads)):
        assert torch.equal(a, b)
