"""The query metric of the EchoSparse representatives (chol_kernel, by panels of 16 columns) against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _metric(q):
    """metric_t [H, 128, 128] (row j = column j of the Cholesky factor) left in the build's workspace."""
    from self_trainable_or_free_attn_amd.kernels import gfx950 as K
    L, H, D = q.shape
    reps = K.Representatives(L, H, D, q.device)
    k = torch.randn(q.shape, device=q.device).bfloat16()
    reps.build(q, k, k)
    rows = -(-(-(-L // 16)) // 64) * 64               # rows of one Gram split
    gram_bytes = H * -(-L // rows) * D * D * 4
    return reps._ws[gram_bytes:gram_bytes + H * D * D * 2].view(torch.bfloat16).view(H, D, D)


@pytest.mark.parametrize("kind", ["full", "low_rank", "one_direction", "one_channel"])
def test_metric_matches_float64_cholesky(kind):
    L, H, D = 4152, 3, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)
    q = {"full": lambda: rand(L, H, D),
         "low_rank": lambda: torch.einsum("lr,hrd->lhd", rand(L, 17), rand(H, 17, D)),   # ends inside a panel
         "one_direction": lambda: rand(1, H, D).expand(L, H, D) + 1e-3 * rand(L, H, D),
         "one_channel": lambda: rand(L, H, D) * (torch.arange(D, device="cuda") == 15)}[kind]().bfloat16()
    got = _metric(q).double()
    x = q.double().permute(1, 0, 2)
    G = x.transpose(1, 2) @ x / (D * L)
    G = G + 1e-3 * G.diagonal(dim1=1, dim2=2).mean(1)[:, None, None] * torch.eye(D, device="cuda")
    want = torch.linalg.cholesky(G).transpose(1, 2)
    # half a bf16 step of each entry, and the float32 factorisation: the ridge (1e-3 of the mean diagonal) bounds the
    # cancellation of a pivot, so its error is at most about 128 * 2^-24 / 1e-3 of the factor's largest entry
    bound = 2 ** -8 * want.abs() + 1e-2 * 2 ** -7 * want.abs().amax((1, 2), keepdim=True)
    err = (got - want).abs()
    print(kind, "max err / bound", float((err / bound).max()))
    assert bool((err <= bound).all())
    assert bool((got.tril(-1) == 0).all())
