"""How the VSA operators hand D = 64 rows to the entry points, which read D columns of every row whatever the tensor's
width: fake GPU tensors, nothing is launched."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from self_trainable_or_free_attn_amd import _lib
from self_trainable_or_free_attn_amd.vsa import _C

BF = torch.bfloat16


def test_rows_pad_and_narrow():
    x = torch.arange(1, 97.0).view(3, 32)
    assert torch.equal(_C._rows(x, 64), torch.cat([x, torch.zeros(3, 32)], 1))
    y = torch.arange(1, 301.0).view(3, 100)
    assert torch.equal(_C._rows(y, 64), y[:, :64]) and _C._rows(y, 64).is_contiguous()
    assert torch.equal(_C._rows(x, 128), torch.cat([x, torch.zeros(3, 96)], 1))


@pytest.mark.parametrize("width", [16, 32, 63, 64, 100, 128])
def test_secondary_tensors_reach_the_kernels_with_full_rows(monkeypatch, width):
    """A coarse output, a gradient to add and a partial of another width than the tokens' 64."""
    calls = []
    monkeypatch.setattr(_lib, "call", lambda name, *args: calls.append((name, args)))
    with FakeTensorMode():
        tok = lambda w=64: torch.empty(1, 2, 320, w, device="cuda", dtype=BF)
        f32 = lambda *s: torch.empty(*s, device="cuda")
        cnt = torch.empty(5, device="cuda", dtype=torch.int32)
        oc, add = torch.empty(1, 2, 64, width, device="cuda", dtype=BF), f32(1, 2, 64, width)
        _C.fuse_fwd(tok(), oc, None, cnt, 0)
        _C.fuse_bwd(tok(), tok(width), oc, None, cnt, 0)
        _C.finalize(f32(1, 2, 320, width), add, cnt, tok())
        _C.row_dot(tok(), tok(width), cnt)
        i32 = lambda *s: torch.empty(*s, device="cuda", dtype=torch.int32)
        _C.split_merge_sum(f32(4, 64, width), i32(2, 4), i32(8), add, cnt, tok())
        _C.router_lse(torch.empty(1, 2, 64, 64, device="cuda", dtype=BF), oc, cnt, 16)
        _C.attn_bwd_q(tok(), tok(), tok(), tok(width), f32(1, 2, 320), f32(1, 2, 320), i32(1, 2, 6), i32(20), cnt, add)
    assert len(calls) == 7
    for name, args in calls:
        for a in args:                     # (the float tensors that are not per-token statistics, [1, 2, 320])
            if isinstance(a, torch.Tensor) and a.is_floating_point() and a.shape[-1] != 320:
                assert a.shape[-1] == 64 and a.is_contiguous(), (name, tuple(a.shape))


def _fine(q, k, v, cnt, a, b, c, d):
    from self_trainable_or_free_attn_amd.vsa import Selection, fine_block_sparse_attention
    return fine_block_sparse_attention(q, k, v, cnt, Selection(a, b, c, d), backend="generic")


def _fine_args(D):
    i32 = lambda *s: torch.empty(*s, device="cuda", dtype=torch.int32)
    qkv = [torch.empty(1, 2, 320, D, device="cuda", dtype=BF) for _ in range(3)]
    return (*qkv, i32(5), i32(1, 2, 6), i32(20), i32(1, 2, 6), i32(20))


TRACED = {
    "fine_block_sparse_attention": (_fine, _fine_args),
    "attn_fwd": (lambda q, k, v, cnt, a, b, c, d: _C.attn_fwd(q, k, v, a, b, cnt), _fine_args),
    "attn_bwd_q_acc": (lambda q, k, v, cnt, a, b, c, d: _C.attn_bwd_q_acc(
        q, k, v, q, q[..., 0].float(), q[..., 0].float(), a, b, cnt, q.float()), _fine_args),
    "pool_fwd": (lambda q, k, v, cnt, a, b, c, d: _C.pool_fwd(q, k, v, cnt, 16), _fine_args),
    "row_dot": (lambda q, k, v, cnt, a, b, c, d: _C.row_dot(q, k, cnt), _fine_args),
}


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("name", sorted(TRACED))
def test_operators_trace_into_one_graph(name, dynamic, D):
    """Under torch.compile(fullgraph=True) a tensor has no address to look at."""
    f, args = TRACED[name]
    _lib.ops()
    torch._dynamo.reset()
    with FakeTensorMode(allow_non_fake_inputs=True):
        out = torch.compile(f, fullgraph=True, backend="eager", dynamic=dynamic)(*args(D))
    first = out[0] if isinstance(out, (list, tuple)) else out
    assert first.is_cuda and first.shape[:2] == (1, 2)


@pytest.mark.parametrize("D", [64, 128])
def test_operators_under_forward_mode(D):
    """A torch.func wrapper is a torch.Tensor without storage; the operators have no derivative, and take it."""
    with FakeTensorMode(allow_non_fake_inputs=True):
        q, k, v, cnt, *lists = _fine_args(D)
        (o, lse), _ = torch.func.jvp(lambda x: _C.attn_fwd(x, k, v, *lists[:2], cnt), (q,), (torch.ones_like(q),))
        assert o.shape == q.shape and lse.shape == q.shape[:3]
        dot, _ = torch.func.jvp(lambda x: _C.row_dot(x, k, cnt), (q,), (torch.ones_like(q),))
        assert dot.shape == q.shape[:3]


def test_unaligned_rows_are_copied():
    x = torch.zeros(3 * 64 + 1, dtype=BF)
    aligned, shifted = x[:-1].view(3, 64), x[1:].view(3, 64)
    assert _C._rows(aligned, 64) is aligned
    copy = _C._rows(shifted, 64)
    assert copy is not shifted and copy.data_ptr() % 16 == 0 and torch.equal(copy, shifted)


@pytest.mark.parametrize("phases", range(8))
def test_table_gradients_pad_only_the_tables_in_use(monkeypatch, phases):
    """At D = 64 a table's gradients are padded to 128 columns and written back: only those of the tiers that run."""
    calls, wide = [], []
    monkeypatch.setattr(_lib, "call", lambda name, *args: calls.append(name))
    pad = _C._wide
    monkeypatch.setattr(_C, "_wide", lambda x: wide.append(x) or pad(x))
    with FakeTensorMode():
        bf = lambda n, w=64: torch.empty(1, 2, n, w, device="cuda", dtype=BF)
        f32, i32 = (lambda *s, t=t: torch.empty(*s, device="cuda", dtype=t) for t in (torch.float32, torch.int32))
        grads = [f32(1, 2, n, 64) for n in (64, 64, 64, 64)]
        _C.rep_attn_bwd_q(bf(320), bf(320), bf(320), bf(64), bf(64), f32(20), bf(64), bf(64), f32(5), bf(320),
                          f32(1, 2, 320), f32(1, 2, 320), i32(1, 2, 6), i32(20), i32(1, 2, 5, 1), i32(1, 2, 5, 1),
                          i32(5), *grads, 4, phases)
    used = (grads[:2] if phases & 2 else []) + (grads[2:] if phases & 4 else [])
    seen = [x for x in wide if any(x is g for g in grads)]
    assert len(seen) == len(used) and all(any(x is g for x in seen) for g in used)
    want = {0: [], 2: ["vsa_rep_bwd_tables"], 4: ["vsa_rep_bwd_tables"], 6: ["vsa_rep_bwd_both_tables"]}[phases & 6]
    assert calls[1:] == want
