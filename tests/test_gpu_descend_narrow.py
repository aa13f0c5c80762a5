"""The two forms of the descent of many queries -- a beam of at most 8 over a binary tree (a 16-lane group per query), and
wide beams whose kept set is found without ranking -- against the oracle's canonical descent, bit for bit.  GPU only."""
import pytest
import torch

from oracle import seg_ref as S
from treeattn_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = 'cuda'


@pytest.mark.parametrize('T,D,leaf,wmax,Nq,dtype', [
    (1024, 64, 2, 8, 257, torch.float16),     # the fewest queries; a last group of one query
    (4096, 128, 2, 8, 300, torch.float32),
    (4096, 128, 2, 8, 515, torch.float32),    # candidate rows in three parts (from 1024 queries on)
    (1024, 64, 2, 8, 5, torch.float32),       # the fewest queries a pair
    (512, 16, 2, 1, 512, torch.bfloat16),     # a beam of one
    (256, 32, 2, 5, 256, torch.float32),      # every position, an odd beam
    (64, 64, 32, 8, 64, torch.bfloat16),      # one level
    (2048, 64, 16, 7, 1000, torch.bfloat16),
])
def test_narrow_descent_matches_oracle(T, D, leaf, wmax, Nq, dtype):
    print('case', T, D, leaf, wmax, Nq, dtype, flush=True)
    B, H = (3, 2) if 5 < Nq < 300 else (60, 9) if Nq == 5 else (1, 2)
    g = torch.Generator().manual_seed(T + D + wmax)
    q = torch.randn(B, H, Nq, D, generator=g).to(dtype)
    k = torch.randn(B, H, T, D, generator=g).to(dtype)
    k[:, :, T // 2:] = k[:, :, :T // 2]       # repeated keys: equal scores, ranked by node id
    # sorted positions from 0 on, some repeated, the last one included: starts differ within a wavefront
    tq = torch.arange(T) if Nq == T else torch.sort(torch.randint(0, T, (Nq,), generator=g)).values
    tq[-1] = T - 1
    geom = S.Geometry(T, leaf, 2)
    want = S.tree_pass_general(q.float(), S.pyramid(S.index_keys(k), geom), tq, geom, wmax, 'canonical')
    shape = K.TreeShape(T, leaf, 2)
    lv = K.level_sums(k.to(DEV), shape.blevels)
    NS = 3
    store = (torch.full((B, H, T, NS), -7, dtype=torch.int32, device=DEV), torch.full((B, H, T, NS), 7.0, device=DEV),
             torch.ones(B, H, T, NS, dtype=torch.bool, device=DEV))
    n = min(NS, shape.leaf_width(wmax))
    ids, vld, sct = (x.cpu() for x in K.tree_descend(q.to(DEV), lv, tq.to(DEV), shape, wmax, store=(*store, n)))
    ok = want[1]
    assert torch.equal(vld.bool(), ok)
    assert torch.equal(ids.long()[ok], want[0][ok]) and torch.equal(sct[ok], want[2][ok])
    assert bool((ids[~ok] == -1).all())
    sl, ss, so = (x.cpu() for x in store)
    rows = tq.unique()                        # a repeated position is written by any of its (different) queries
    once = [int(i) for i in rows if int((tq == i).sum()) == 1]
    at = torch.tensor([int((tq == i).nonzero()[0]) for i in once])
    w_ok = ok[:, :, at, :n]
    assert torch.equal(so[:, :, once, :n], w_ok)
    assert torch.equal(sl[:, :, once, :n].long(), torch.where(w_ok, want[0][:, :, at, :n], 0))
    assert torch.equal(ss[:, :, once, :n], torch.where(w_ok, want[2][:, :, at, :n], 0.0))
    assert bool((sl[..., n:] == -7).all())


@pytest.mark.parametrize('T,D,leaf,arity,wmax,copies', [
    (8192, 64, 32, 2, 32, 1),      # 64 and 65 candidates
    (8192, 64, 32, 2, 32, 16),     # equal scores at the border of the kept set
    (2048, 16, 16, 4, 31, 1),      # up to 127 candidates, a beam that is no multiple of 4
    (4096, 32, 32, 2, 64, 4),      # 128 and 129 candidates: both sides of what one wavefront holds
])
def test_wide_descent_matches_oracle(T, D, leaf, arity, wmax, copies):
    print('case', T, D, leaf, arity, wmax, copies, flush=True)
    B, H, Nq = 1, 2, 2200
    g = torch.Generator().manual_seed(T + D + wmax)
    q = torch.randn(B, H, Nq, D, generator=g)
    k = torch.randn(B, H, T // copies, D, generator=g).repeat(1, 1, copies, 1)
    tq = torch.sort(torch.randint(0, T, (Nq,), generator=g)).values
    geom = S.Geometry(T, leaf, arity)
    want = S.tree_pass_general(q, S.pyramid(S.index_keys(k), geom), tq, geom, wmax, 'canonical')
    shape = K.TreeShape(T, leaf, arity)
    lv = K.level_sums(k.to(DEV), shape.blevels)
    ids, vld, sct = (x.cpu() for x in K.tree_descend(q.to(DEV), lv, tq.to(DEV), shape, wmax))
    ok = want[1]
    assert torch.equal(vld.bool(), ok)
    assert torch.equal(ids.long()[ok], want[0][ok]) and torch.equal(sct[ok], want[2][ok])


def _us(f):
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = float('inf')
    for _ in range(6):
        a.record()
        for _ in range(8):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1000 / 8)
    return best


def test_few_queries_per_pair_keep_their_wavefronts():
    """One query of each of 2048 (sequence, head) pairs at D = 128, as a decode step asks: with a 16-lane group per query,
    15 of a workgroup's 16 idle, this took 1.9 times the wavefronts per query, which a beam of 9 still takes."""
    T, D, w = 4096, 128, 8
    shape = K.TreeShape(T, 2, 2)
    g = torch.Generator(device=DEV).manual_seed(1)
    k = torch.randn(1, 4, T, D, generator=g, device=DEV)
    lv = [x.expand(512, 4, -1, -1) for x in K.level_sums(k, shape.blevels)]
    q = torch.randn(512, 4, 1, D, generator=g, device=DEV)
    tq = torch.tensor([T - 5], dtype=torch.int32, device=DEV)
    out = K.tree_descend(q, lv, tq, shape, w)
    few = _us(lambda: K.tree_descend(q, lv, tq, shape, w, out=out))
    # a beam of 9 is past the 16-lane groups: the same work by wavefronts, a ninth more of it
    out9 = K.tree_descend(q, lv, tq, shape, 9)
    assert few < 1.25 * _us(lambda: K.tree_descend(q, lv, tq, shape, 9, out=out9))
