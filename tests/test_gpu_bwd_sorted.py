"""The sorted dk / dv route of ta_sparse_attn_bwd at the sizes where its sort and its row handling can go wrong,
against the closed form in float64.  GPU only."""
import math

import pytest
import torch

from treeattn_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _backward64(q, k, v, cand, scale, do):
    """out, lse, dq, dk, dv of softmax attention over the candidate rows, float64."""
    q, k, v, do = [x.double() for x in (q, k, v, do)]
    B, H, T, D = q.shape
    Tk = k.shape[2]
    ok = (cand >= 0) & (cand < Tk)
    out, lse = torch.zeros_like(q), torch.zeros(B, H, T, dtype=torch.float64)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for b in range(B):
        for h in range(H):
            idx = torch.where(ok[b, h], cand[b, h], 0)
            kg, vg = k[b, h][idx], v[b, h][idx]
            s = ((q[b, h].unsqueeze(1) * kg).sum(-1) * scale).masked_fill(~ok[b, h], -math.inf)
            p = torch.softmax(s, -1)
            out[b, h], lse[b, h] = (p.unsqueeze(-1) * vg).sum(1), torch.logsumexp(s, -1)
            dp = (do[b, h].unsqueeze(1) * vg).sum(-1)
            ds = p * (dp - (p * dp).sum(-1, keepdim=True))
            dq[b, h] = scale * (ds.unsqueeze(-1) * kg).sum(1)
            dk[b, h].index_add_(0, idx.reshape(-1), (scale * ds.unsqueeze(-1) * q[b, h].unsqueeze(1)).reshape(-1, D))
            dv[b, h].index_add_(0, idx.reshape(-1), (p.unsqueeze(-1) * do[b, h].unsqueeze(1)).reshape(-1, D))
    return out, lse, dq, dk, dv


@pytest.mark.parametrize('T,Tk,KC,D,misaligned', [
    (1, 1, 1, 8, False),           # one slot
    (65, 63, 9, 24, False),        # lanes past the row, keys short of a bucket, slots past the last key
    (2600, 2600, 12, 64, False),   # a key with more entries than one LDS tile
    (300, 300, 70, 256, False),    # a wavefront's half per row
    (40, 140000, 11, 8, False),    # buckets of more than 64 keys
    (3, 500, 4200, 16, False),     # a chunk of one query, a query naming a key many times
    (130, 130, 33, 40, True),      # rows that are not 16-byte aligned
])
def test_sorted_backward_matches_float64(T, Tk, KC, D, misaligned):
    print('case', T, Tk, KC, D, misaligned, flush=True)
    B, H = 2, 2
    g = torch.Generator().manual_seed(T + KC)
    q, do = (torch.randn(B, H, T, D, generator=g) for _ in range(2))
    k, v = (torch.randn(B, H, Tk, D, generator=g) for _ in range(2))
    cand = torch.randint(-2, Tk + 2, (B, H, T, KC), generator=g)
    cand[..., 0] = 0               # a key every query names
    scale = 1 / math.sqrt(D)
    qd, kd, vd, cd, dd = (x.to(DEV) for x in (q, k, v, cand, do))
    if misaligned:
        qd = torch.cat([qd.new_zeros(1), qd.reshape(-1)])[1:].view(B, H, T, D)
        dd = torch.cat([dd.new_zeros(1), dd.reshape(-1)])[1:].view(B, H, T, D)
        assert qd.data_ptr() % 16 and dd.data_ptr() % 16
    out, lse, *want = _backward64(q, k, v, cand, scale, do)
    out, lse = out.float().to(DEV), lse.float().to(DEV)
    got = K.sparse_attn_bwd(qd, kd, vd, cd, scale, out, lse, dd, deterministic=True)
    again = K.sparse_attn_bwd(qd, kd, vd, cd, scale, out, lse, dd, deterministic=True)
    # float32 sums of n terms: an error of about sqrt(n) * 2^-24 of the terms' norm; 1e-5 of the largest value is
    # above that for the 2600 terms of the key that every query names
    for a, b, w in zip(got, again, want):
        assert torch.equal(a, b)
        assert (a.cpu().double() - w).abs().max().item() <= 1e-5 * max(1.0, w.abs().max().item())


@pytest.mark.parametrize('T,Tk,KC', [
    ((1 << 22) + 5, 300, 2),       # more queries than an entry can name: sorted in two parts
    (20000, (1 << 21) + 33, 6),    # more keys than the buckets hold: summed in two parts
    (16400, 5000, 4100),           # more slots than the workspace holds at a time, a chunk per query
])
def test_fixed_order_past_one_sort(T, Tk, KC):
    """Sizes whose slots are sorted in several parts: the same bits every time (a key that every query names would
    show another order), and the closed form in float64."""
    print('case', T, Tk, KC, flush=True)
    D, scale = 8, 1 / math.sqrt(8)
    g = torch.Generator().manual_seed(T + KC)
    q, do = (torch.randn(1, 1, T, D, generator=g) for _ in range(2))
    k, v = (torch.randn(1, 1, Tk, D, generator=g) for _ in range(2))
    cand = torch.randint(-2, Tk + 2, (1, 1, T, min(KC, 30)), generator=g)   # the slots after those are unused
    cand[..., 0] = 0
    out, lse, *want = _backward64(q, k, v, cand, scale, do)
    q, k, v, do, out, lse = (x.float().to(DEV) for x in (q, k, v, do, out, lse))
    cand = torch.nn.functional.pad(cand.int().to(DEV), (0, KC - cand.shape[-1]), value=-1)
    got = K.sparse_attn_bwd(q, k, v, cand, scale, out, lse, do, deterministic=True)
    again = K.sparse_attn_bwd(q, k, v, cand, scale, out, lse, do, deterministic=True)
    # a key's list is added in up to 2050 parts (one per tile of 2048 entries) whose running sum is rounded each time:
    # about sqrt(2050) * 2^-24 = 2.7e-6 of the largest value
    for a, b, w in zip(got, again, want):
        assert torch.equal(a, b)
        assert (a.cpu().double() - w).abs().max().item() <= 1e-5 * max(1.0, w.abs().max().item())


def test_pairs_in_groups_equal_pairs_alone():
    """More slots than the workspace holds at a time, over the (sequence, head) pairs: each pair's gradients are bit for
    bit those of a call on it alone."""
    B, H, T, D, KC = 1, 36, 500, 8, 4000
    g = torch.Generator(device=DEV).manual_seed(9)
    q, k, v, do, out = (torch.randn(B, H, T, D, generator=g, device=DEV) for _ in range(5))
    cand = torch.randint(-3 * T, T, (B, H, T, KC), generator=g, device=DEV, dtype=torch.int32)
    lse = torch.full((B, H, T), 7.0, device=DEV)   # any values do: what is compared is the same sums
    got = K.sparse_attn_bwd(q, k, v, cand, 0.3, out, lse, do, deterministic=True)
    for h in (0, 28, 29, 35):   # 29 pairs are sorted together
        part = [x[:, h:h + 1] for x in (q, k, v, cand, out, lse, do)]
        alone = K.sparse_attn_bwd(*part[:4], 0.3, *part[4:], deterministic=True)
        assert all(torch.equal(a[:, h:h + 1], b) for a, b in zip(got, alone))


def test_no_slots_with_a_workspace_gives_zeros():
    """No candidate slots: dq, dk and dv are written as zeros (the entry point itself; the wrapper takes no workspace)."""
    from treeattn_amd import _lib as L
    B, H, T, Tk, D = 2, 3, 5, 700, 24
    q, o, do = (torch.randn(B, H, T, D, device=DEV) for _ in range(3))
    k, v = (torch.randn(B, H, Tk, D, device=DEV) for _ in range(2))
    dq, dk, dv = (torch.full_like(x, 7.0) for x in (q, k, v))
    cand, ws = torch.zeros(1, dtype=torch.int32, device=DEV), torch.zeros(4, device=DEV)
    lse = torch.zeros(B, H, T, device=DEV)
    L.call('ta_sparse_attn_bwd', *(L.ptr(x) for x in (q, k, v, o, do)), L.F32, *L.rows3(q), *L.rows3(k), *L.rows3(v),
           *L.rows3(o), *L.rows3(do), L.ptr(cand), L.ptr(lse), B, H, T, Tk, 0, D, 1.0, L.ptr(dq), L.ptr(dk), L.ptr(dv),
           L.ptr(ws), 0, L.stream())
    assert all(bool((x == 0).all()) for x in (dq, dk, dv))


@pytest.mark.parametrize('dtype,T,H,D', [(torch.float32, 130, 3, 16), (torch.float16, 77, 2, 64), (torch.bfloat16, 1, 2, 128),
                                         (torch.float16, 33, 1, 64), (torch.float16, 50, 2, 32)])
@pytest.mark.parametrize('case', ['views', 'offset', 'broadcast'])
def test_strided_rows_equal_contiguous(dtype, T, H, D, case):
    """q, k and v as views of one projection (read in place, gradients laid out alike), such views off 16-byte alignment
    and a broadcast gradient of the output: bit for bit the contiguous tensors' results."""
    B, KC = 2, 9
    g = torch.Generator().manual_seed(T)
    n = B * T * 3 * H * D
    flat = torch.randn(n + 1, generator=g).to(dtype).to(DEV)
    qkv = (flat[1:] if case == 'offset' else flat[:n]).view(B, T, 3 * H * D)
    q, k, v = (t.view(B, T, H, D).transpose(1, 2) for t in qkv.split(H * D, dim=2))
    do = torch.randn(B, T, H, D, generator=g).to(dtype).to(DEV).transpose(1, 2)
    if case == 'broadcast':
        do = do[:, :1, :1, :1].expand(B, H, T, D)
    cand = torch.randint(-1, T, (B, H, T, KC), generator=g).to(DEV)
    c = [t.contiguous() for t in (q, k, v, do)]
    out, lse = K.sparse_attn_fwd(*c[:3], cand, 0.125)
    want = K.sparse_attn_bwd(*c[:3], cand, 0.125, out, lse, c[3], deterministic=True)
    got = K.sparse_attn_bwd(q, k, v, cand, 0.125, out, lse, do, deterministic=True)
    assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(got, want))
    # atomic adds: float32 sums of up to T KC terms in any order, rounded to the type
    tol = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype]
    for a, b in zip(K.sparse_attn_bwd(q, k, v, cand, 0.125, out, lse, do, deterministic=False), want):
        assert (a.float() - b.float()).abs().max().item() <= tol * max(1.0, b.float().abs().max().item())


def test_workspace_off_alignment():
    """A workspace aligned to float32 only: the same bits, and nothing past its size is written."""
    from treeattn_amd import _lib as L
    B, H, T, KC, D = 1, 2, 90, 7, 16
    g = torch.Generator().manual_seed(4)
    q, k, v, o, do = (torch.randn(B, H, T, D, generator=g).to(DEV) for _ in range(5))
    cand = torch.randint(-1, T, (B, H, T, KC), generator=g, dtype=torch.int32).to(DEV)
    lse = torch.full((B, H, T), 2.0, device=DEV)
    words = L.lib().ta_sparse_attn_bwd_workspace_size(B, H, T, KC) // 4
    got = []
    for off in (0, 1):
        buf = torch.full((words + 4,), 7.0, device=DEV)
        assert buf.data_ptr() % 8 == 0
        grads = [torch.empty(B, H, T, D, device=DEV) for _ in range(3)]
        L.call('ta_sparse_attn_bwd', *(L.ptr(x) for x in (q, k, v, o, do)), L.F32,
               *(s for x in (q, k, v, o, do) for s in L.rows3(x)), L.ptr(cand), L.ptr(lse), B, H, T, T, KC, D, 1.0,
               *(L.ptr(x) for x in grads), L.ptr(buf[off:]), 0, L.stream())
        assert bool((buf[off + words:] == 7).all())
        got.append(grads)
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize('T,D,dtype', [(1, 8, torch.float32), (70, 64, torch.float16), (33, 24, torch.bfloat16)])
def test_contiguous_keys_off_alignment(T, D, dtype):
    """Contiguous keys and values off a 16-byte boundary, and a single pair with an odd stride of its batch: the bits of
    the aligned ones."""
    g = torch.Generator().manual_seed(T)
    q, k, v, do, out = (torch.randn(1, 1, T, D, generator=g).to(dtype).to(DEV) for _ in range(5))
    cand = torch.randint(-1, T, (1, 1, T, 9), generator=g).to(DEV)
    lse = torch.zeros(1, 1, T, device=DEV)
    want = K.sparse_attn_bwd(q, k, v, cand, 0.1, out, lse, do)
    off = [torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(1, 1, T, D) for x in (k, v)]
    odd = [x.as_strided((1, 1, T, D), (3, 5, D, 1)) for x in (k, v)]
    for kv in (off, odd):
        assert kv[0].is_contiguous()
        assert all(torch.equal(a, b) for a, b in zip(K.sparse_attn_bwd(q, *kv, cand, 0.1, out, lse, do), want))


def test_atomic_route_adds_whole_lines():
    """The atomic adds go to consecutive dimensions from consecutive lanes: with lanes 32 bytes apart this call took 13.4
    times the sorted route's, with consecutive ones 1.8 times."""
    B, H, T, D, KC = 2, 6, 2048, 64, 13
    g = torch.Generator(device=DEV).manual_seed(5)
    q, k, v, do = (torch.randn(B, H, T, D, generator=g, device=DEV) for _ in range(4))
    cand = torch.randint(0, T, (B, H, T, KC), generator=g, device=DEV, dtype=torch.int32)
    out, lse = K.sparse_attn_fwd(q, k, v, cand, 0.125)

    def us(det):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = math.inf
        for _ in range(6):
            a.record()
            for _ in range(4):
                K.sparse_attn_bwd(q, k, v, cand, 0.125, out, lse, do, deterministic=det)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best
    assert us(False) < 9 * us(True)


def test_default_is_the_fixed_order_at_training_lengths():
    """The default at a long training sequence: the fixed order's bits (atomic adds to the key that every query names
    would differ between runs)."""
    B, H, T, D, KC = 1, 6, 32768, 64, 52
    g = torch.Generator(device=DEV).manual_seed(6)
    q, k, v, do = (torch.randn(B, H, T, D, generator=g, device=DEV) for _ in range(4))
    cand = torch.randint(-3 * T, T, (B, H, T, KC), generator=g, device=DEV, dtype=torch.int32)
    cand[..., 0] = 0
    out, lse = K.sparse_attn_fwd(q, k, v, cand, 0.125)
    got = K.sparse_attn_bwd(q, k, v, cand, 0.125, out, lse, do)
    for det in (None, True):
        again = K.sparse_attn_bwd(q, k, v, cand, 0.125, out, lse, do, deterministic=det)
        assert all(torch.equal(a, b) for a, b in zip(got, again))
