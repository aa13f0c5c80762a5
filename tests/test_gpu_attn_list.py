"""Attention over candidate lists: list lengths around the 64 and 256 slots the kernel packs at a time, dense and
nearly empty lists, every row width, and rows that no slot chose holding infinities."""
import math

import pytest
import torch

from oracle.attn_ref import sparse_attn_lse, sparse_attn_ref

pytestmark = pytest.mark.gpu
DEV = 'cuda'
# the softmax weights and sums are float32 (1e-6 of values of order 1); the result is rounded to its type
TOL = {torch.float32: 1e-5, torch.float16: 4e-3, torch.bfloat16: 3e-2}


@pytest.mark.parametrize('dtype,D', [(torch.float32, 16), (torch.float32, 32), (torch.float32, 128),
                                     (torch.float16, 16), (torch.float16, 32), (torch.float16, 64),
                                     (torch.bfloat16, 128)])
@pytest.mark.parametrize('KC', [1, 63, 65, 256, 257, 530])
def test_attn_list_sizes(dtype, D, KC):
    from treeattn_amd import kernels as K
    B, H, T, Tk = 1, 2, 37, 400
    g = torch.Generator().manual_seed(KC)
    q = torch.randn(B, H, T, D, generator=g).to(dtype)
    k, v = (torch.randn(B, H, Tk, D, generator=g).to(dtype) for _ in range(2))
    cand = torch.randint(1, Tk, (B, H, T, KC), generator=g)
    share = torch.rand(1, 1, T, 1, generator=g)
    cand[torch.rand(B, H, T, KC, generator=g) > share] = -1
    cand[:, :, 3] = -1                  # a row with nothing valid
    cand[:, :, 4, :-1] = -1             # the last slot alone
    cand[:, :, 4, -1] = Tk - 1
    k[:, :, 0] = v[:, :, 0] = math.inf   # chosen by no slot
    scale = 1 / math.sqrt(D)
    out, lse = K.sparse_attn_fwd(q.to(DEV), k.to(DEV), v.to(DEV), cand.to(DEV), scale)
    k[:, :, 0] = v[:, :, 0] = 0
    want, wl = sparse_attn_ref(q, k, v, cand, scale), sparse_attn_lse(q, k, v, cand, scale)
    assert (out.cpu().float() - want.float()).abs().max().item() < TOL[dtype]
    has = (cand >= 0).any(-1)
    assert (lse.cpu() - wl)[has].abs().max().item() < 1e-5 * max(1.0, wl[has].abs().max().item())
    assert (out.cpu()[~has] == 0).all()
