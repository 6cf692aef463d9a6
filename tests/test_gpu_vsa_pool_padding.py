"""Pooling, table building and the fusion backward write their padding rows: outputs allocated over memory that held
NaN are zero past the last block, and the pooled means equal the oracle's bit for bit at ragged block counts."""
import numpy as np
import pytest
import torch

from helpers import f32
from oracle import vsa_ref as ref

pytestmark = pytest.mark.gpu


def _poison(dev):
    """Leaves NaN in the memory that the next allocations are likely to get."""
    x = [torch.full((1 << 20,), float("nan"), device=dev) for _ in range(16)]
    torch.cuda.synchronize()
    del x


@pytest.mark.parametrize("NB,R", [(1, 4), (3, 8), (45, 16), (63, 32), (65, 4), (64, 16)])
def test_pool_and_fuse_padding_rows(dev, NB, R):
    from self_trainable_or_free_attn_amd.vsa import _C
    B, H, D = 1, 3, 128
    g = torch.Generator().manual_seed(NB + R)
    cnt = torch.randint(1, 65, (NB,), generator=g).to(torch.int32)
    x = torch.randn(B, H, NB * 64, D, generator=g).bfloat16()
    xd, blk = x.to(dev), cnt.to(dev)
    _poison(dev)
    qr, kr, qc, kc, vc = _C.pool_fwd(xd, xd, xd, blk, R)
    G = 64 // R
    want_r, want_c = ref.pool(f32(x), cnt.numpy(), R)
    for got in (qr, kr):
        assert np.array_equal(f32(got)[:, :, :NB * G], np.asarray(want_r)[:, :, :NB * G])
        assert not f32(got)[:, :, NB * G:].any()
    for got in (qc, kc, vc):
        assert np.array_equal(f32(got)[:, :, :NB], np.asarray(want_c)[:, :, :NB])
        assert not f32(got)[:, :, NB:].any()
    _poison(dev)
    tab = _C.rep_build(xd, xd, blk, G)
    for t, rows in ((tab[0], NB * G), (tab[1], NB * G), (tab[3], NB), (tab[4], NB)):
        assert not f32(t)[:, :, rows:].any()
    oc = torch.randn(B, H, (NB + 63) // 64 * 64, D, device=dev).bfloat16()
    _poison(dev)
    _, _, dout_c, delta_c, _ = _C.fuse_bwd(xd, xd, oc, None, blk, 0, False)
    assert not f32(dout_c)[:, :, NB:].any() and not f32(delta_c)[:, :, NB:].any()
