"""ta_assemble_leaves (candidate list, budgets and statistics from a selection's leaves) against the torch expansion and
assembly in treeattn_amd.selection, element for element.  GPU only."""
import pytest
import torch

from treeattn_amd import kernels as K
from treeattn_amd import selection as SEL
from treeattn_amd.config import Config

pytestmark = pytest.mark.gpu
DEV = 'cuda'


@pytest.mark.parametrize('b,H,N,wl,leaf,Wn,NS,local,batched', [
    (2, 3, 64, 8, 2, 8, 2, 3, False), (1, 2, 129, 5, 2, 4, 2, 1, False), (2, 2, 97, 6, 4, 3, 2, 5, True),
    (1, 1, 70, 64, 2, 32, 2, 62, False),     # the widest rows: 64 leaves of each kind, 63 static keys
    (1, 2, 300, 7, 128, 0, 0, 3, False),     # no neighbours, an own leaf group of more than a wavefront
    (1, 1, 1, 1, 16, 1, 1, 3, True),         # one row
    (3, 5, 1100, 3, 2, 2, 3, 3, False),      # more rows than the launch has wavefronts
])
def test_list_budgets_and_sums_equal_the_torch_assembly(b, H, N, wl, leaf, Wn, NS, local, batched):
    print('case', b, H, N, wl, leaf, Wn, NS, local, batched, flush=True)
    g = torch.Generator().manual_seed(N + wl)
    S = Wn * NS
    T = max(N, 4 * leaf)
    t = torch.randint(0, T, (b, N), generator=g) if batched else torch.arange(N)
    tb = (t.view(b, 1, N, 1) if batched else t.view(1, 1, N, 1))
    ids = torch.randint(0, 12, (b, H, N, wl), generator=g)
    vld = (torch.rand(b, H, N, wl, generator=g) < 0.8) & ((ids + 1) * leaf <= tb)
    nid = torch.randint(0, 12, (b, H, N, S), generator=g)
    match = (torch.rand(b, H, N, S, generator=g) < 0.6) & ((nid + 1) * leaf <= tb)
    nL = torch.randint(0, S + 1, (b, H, N), generator=g)
    lhat = torch.randint(-2, wl + 3, (b, H, N), generator=g)
    cfg = Config(local=local, wmax=wl, leaf=leaf, nb_window=max(Wn, 1), nb_store=max(NS, 1))
    bor = (nid.int().to(DEV), match.to(DEV), nL.int().to(DEV)) if S else None
    ids32 = torch.where(vld, ids, -1).int().to(DEV)   # an empty slot as a descent writes it
    vld8 = vld.to(torch.uint8).to(DEV)
    cm, n_tree, means = K.assemble_leaves(ids32, vld8, lhat.to(DEV), cfg, leaf, t.int().to(DEV), bor)
    none, n_tree2, means2 = K.assemble_leaves(ids32, vld8, lhat.to(DEV), cfg, leaf, nb=bor, cand=False)
    nLz = nL if S else torch.zeros_like(nL)
    sel = SEL.finish(torch.where(vld, ids, 0), vld, nid, match, nLz, lhat, cfg, leaf)
    cand, keep, used = SEL.assemble(sel, t, cfg, b, H)
    assert torch.equal(cm.cpu().long(), torch.where(keep, cand, -1))
    assert none is None and torch.equal(n_tree, n_tree2) and torch.equal(n_tree.cpu().long(), sel['n_tree'])
    ntp = leaf * wl
    want = torch.tensor([keep.sum(), keep[..., :ntp].sum(), keep[..., ntp:ntp + leaf * S].sum(), used.sum(), nLz.sum()])
    rows = b * H * N
    assert torch.equal(torch.round(means.cpu().double() * rows).long(), want)
    assert torch.equal(means2[3:], means[3:])


def test_budgets_of_very_large_leaves():
    """Budgets and statistics need no list: leaves of more keys than a list's rows can hold."""
    b, H, N, wl, leaf = 1, 2, 300, 3, 1 << 17
    g = torch.Generator().manual_seed(1)
    vld = torch.rand(b, H, N, wl, generator=g) < 0.7
    ids = torch.where(vld, torch.randint(0, 9, (b, H, N, wl), generator=g), -1)
    lhat = torch.randint(0, wl + 2, (b, H, N), generator=g)
    cfg = Config(wmax=wl, leaf=leaf)
    none, n_tree, means = K.assemble_leaves(ids.int().to(DEV), vld.to(torch.uint8).to(DEV), lhat.to(DEV), cfg, leaf,
                                            cand=False)
    want = SEL.budget_split(torch.zeros_like(lhat), lhat, wl)
    used = (vld & (torch.arange(wl) < want.unsqueeze(-1))).sum()
    assert none is None and torch.equal(n_tree.cpu().long(), want)
    assert int(torch.round(means[3].cpu().double() * b * H * N)) == int(used)


def test_positions_and_budgets_of_other_forms():
    """int64 or strided positions and a budget that is broadcast: the list of the plain ones."""
    b, H, N, wl = 2, 3, 50, 5
    g = torch.Generator().manual_seed(2)
    vld = torch.rand(b, H, N, wl, generator=g) < 0.7
    ids = torch.where(vld, torch.randint(0, 9, (b, H, N, wl), generator=g), -1).int().to(DEV)
    cfg = Config(wmax=wl)
    t = torch.randint(20, 90, (b, 2 * N), generator=g).to(DEV)
    one = torch.full((1, 1, 1), 3, device=DEV)
    args = [ids, vld.to(torch.uint8).to(DEV)]
    want = K.assemble_leaves(*args, one.expand(b, H, N).contiguous(), cfg, 2, t[:, ::2].int().contiguous())
    got = K.assemble_leaves(*args, one, cfg, 2, t[:, ::2])
    assert all(torch.equal(a, b) for a, b in zip(got, want))
