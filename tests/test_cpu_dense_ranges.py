"""Dense attention's workspace rule: the binding's arithmetic against the library's, at the edges of the rule and at
random sizes, and dense attention traced into one graph with fake GPU tensors (a ctypes call cannot be traced)."""
import itertools
import random

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from self_trainable_or_free_attn_amd import _lib
from self_trainable_or_free_attn_amd.attention import dense_attention
from self_trainable_or_free_attn_amd.kernels import gfx950 as K


def test_workspace_rule_matches_the_library():
    want = _lib.lib().es_dense_attention_workspace
    r = random.Random(0)
    queries = [-1, 0, 1, 127, 128, 129, 1280, 1281, 2816, 4096, 4097, 32768, 32769]
    keys = [-5, 0, 1, 448, 449, 512, 513, 704, 705, 960, 961, 1024, 1025, 4096, 4097, 1 << 20]
    sizes = list(itertools.product(queries, keys, [0, 1, 2, 3, 8, 12, 24, 128, 129, 256, 257]))
    sizes += [tuple(int(2 ** r.uniform(0, top)) for top in (16, 20, 9)) for _ in range(20000)]
    for s in sizes:
        assert _lib.dense_workspace_bytes(*s) == want(*s), s


@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("Lq,Lk", [(300, 2048), (2048, 2048), (100, 100), (40000, 512)])
def test_dense_attention_traces_into_one_graph(Lq, Lk, dynamic):
    _lib.ops()
    torch._dynamo.reset()
    with FakeTensorMode(allow_non_fake_inputs=True):
        q, k, v = (torch.empty(1, n, 2, 128, device="cuda", dtype=torch.bfloat16) for n in (Lq, Lk, Lk))
        out = torch.compile(dense_attention, fullgraph=True, backend="eager", dynamic=dynamic)(q, k, v)
        assert out.shape == q.shape
        f = K.dense_attention if Lq == Lk else K.dense_attention_kv
        out, lse = torch.compile(f, fullgraph=True, backend="eager", dynamic=dynamic)(q[0], k[0], v[0])
        assert out.shape == q[0].shape and lse.shape == (-(-Lq // 128) * 128, 2)
