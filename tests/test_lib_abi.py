"""CPU-side checks of the C-ABI library: it is built, loads, and exports every entry point include/treeattn.h
declares (no compute calls: there is no GPU here)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, 'include', 'treeattn.h')


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
    return sorted(set(re.findall(r'\b(ta_[a-z_0-9]+)\s*\(', text)))


def test_header_declares_entry_points():
    names = declared_functions()
    for n in ('ta_level_sums', 'ta_tree_descend', 'ta_gather_dot', 'ta_gather_dot_blocks', 'ta_sparse_attn_fwd',
              'ta_seg_attn_fwd', 'ta_kv_append', 'ta_last_error', 'ta_abi_version'):
        assert n in names


def test_library_exports_every_declared_symbol():
    import torch  # noqa: F401  (the library binds to the HIP runtime torch loads)
    from treeattn_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail('libtreeattn.so is not built (python -m treeattn_amd.build)')
    L = _lib.lib()
    for n in declared_functions():
        assert hasattr(L, n), n
    assert set(_lib.SIGNATURES) == set(declared_functions())
    assert L.ta_abi_version() == 3


def test_build_entry_checks_the_declared_abi_version():
    """__graft_entry__.build() compares the library's ABI version with the one include/treeattn.h declares (no
    number of its own to fall behind the header); the built library matches it."""
    import torch  # noqa: F401
    from treeattn_amd import _lib
    src = open(os.path.join(ROOT, '__graft_entry__.py')).read()
    assert 'TA_ABI_VERSION' in src and 'ta_abi_version() == ' not in src
    declared = int(re.search(r'#define TA_ABI_VERSION (\d+)', open(HEADER).read()).group(1))
    assert _lib.lib().ta_abi_version() == declared


def test_library_rejects_bad_arguments_without_gpu():
    """Argument validation runs on the host: a bad size returns an error code and a message."""
    import torch  # noqa: F401
    from treeattn_amd import _lib
    L = _lib.lib()
    rc = L.ta_tree_descend(None, 0, 0, 0, 0, 1, 1, 4, 64, None, 0, 0, None, None, None, 100, 1, 1, 4, 4,
                           None, None, None, None)
    assert rc == 1
    assert b'bad sizes' in L.ta_last_error()
    rc = L.ta_seg_attn_fwd(None, None, None, 2, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 64, 64, None, 0, None, None, None, 4,
                           64, 200, 0.1, None, 0, 0, 0, None, None, 1, None, 0, None, None)
    assert rc == 2
    assert b'local window' in L.ta_last_error()
    # candidate rows wider than 320 entries (leaf 4 x 64 leaves + 128 neighbour keys + 4 static keys + 4 own keys)
    import ctypes
    one = ctypes.c_void_p(8)   # never dereferenced: the sizes are refused first
    rc = L.ta_assemble_candidates(one, one, one, one, one, 0, 1, 1, 8, 64, 4, 128, 3, one, one, None)
    assert rc == 1
    assert b'at most 320 candidates' in L.ta_last_error()
    # the list from leaves: leaves of at most 65536 keys (positions are found in float32), 64 leaves of each kind; the
    # wrapper's callers take the torch assembly where its rule says so
    from treeattn_amd import kernels as K
    for wl, leaf, S, local in [(4, 131072, 0, 3), (65, 2, 0, 3), (4, 2, 65, 3), (4, 2, 16, 64)]:
        assert not K.leaves_supported(wl, leaf, S, local)
        rc = L.ta_assemble_leaves(one, one, one, one, one, one, one, 0, 1, 1, 8, wl, S, leaf, local, wl, one, one, one,
                                  1, None)
        assert rc == 1 and b'at most 65536 for the list' in L.ta_last_error()
    assert K.leaves_supported(64, 65536, 64, 63) and K.leaves_supported(4, 1 << 20, 0, 3, cand=False)
    # LaneTree workspace: T a power of two in [4, 262144], chunk dividing T, head size 16 / 32 / 64 / 128
    nb = ctypes.c_int64(0)
    assert L.ta_lanetree_workspace_size(1, 6, 131072, 64, 4096, ctypes.byref(nb)) == 0
    assert nb.value == 6 * 32 * 131072 * (64 * 4 + 8)
    assert L.ta_lanetree_workspace_size(2, 3, 4096, 128, 64, ctypes.byref(nb)) == 0
    assert nb.value == 2 * 3 * 64 * 4096 * (128 * 4 + 8)
    for bad in [(1, 1, 100, 64, 4), (1, 1, 524288, 64, 4096), (1, 1, 4096, 48, 64), (1, 1, 4096, 64, 48),
                (1, 1, 2, 16, 1), (0, 1, 4096, 64, 64)]:
        assert L.ta_lanetree_workspace_size(*bad, ctypes.byref(nb)) == 1, bad
        assert b'ta_lanetree_workspace_size' in L.ta_last_error()


def test_product_refuses_cpu_tensors():
    import torch
    from treeattn_amd import kernels
    q = torch.zeros(1, 1, 4, 64)
    with pytest.raises(RuntimeError, match='GPU'):
        kernels.gather_dot(q, q, torch.zeros(1, 1, 4, 2, dtype=torch.long), 1.0)


def test_assemble_leaves_checks_its_tensors():
    """Tensors whose memory would be read as something else, or past its end, are refused before any launch."""
    import torch
    from treeattn_amd import kernels as K
    from treeattn_amd.config import Config
    b, H, N, wl, S = 1, 2, 8, 3, 4
    ids, vld = torch.zeros(b, H, N, wl, dtype=torch.int32), torch.zeros(b, H, N, wl, dtype=torch.uint8)
    nb = [torch.zeros(b, H, N, S, dtype=torch.int32), torch.zeros(b, H, N, S, dtype=torch.bool),
          torch.zeros(b, H, N, dtype=torch.int32)]
    lhat, tq = torch.ones(b, H, N, dtype=torch.long), torch.arange(N)

    def call(ids=ids, vld=vld, lhat=lhat, tq=tq, nb=nb):
        K.assemble_leaves(ids, vld, lhat, Config(wmax=wl), 2, tq, nb)
    with pytest.raises(RuntimeError, match='GPU'):   # all in order but for the device
        call()
    wide = torch.zeros(b, H, N, 2 * wl, dtype=torch.int32)
    for bad in (dict(ids=ids.long()), dict(ids=wide[..., ::2]), dict(ids=ids.transpose(1, 2)), dict(vld=vld.bool()),
                dict(vld=vld[:, :, :4]), dict(nb=[nb[0].long(), *nb[1:]]), dict(nb=[nb[0], nb[1].to(torch.uint8), nb[2]]),
                dict(nb=[*nb[:2], nb[2].long()]), dict(nb=[*nb[:2], nb[2][..., :4]])):
        with pytest.raises(TypeError):
            call(**bad)
    for tq in (None, torch.arange(N - 1), torch.zeros(b, H, N)):
        with pytest.raises(ValueError):
            call(tq=tq)
    with pytest.raises(RuntimeError, match='expand'):
        call(lhat=lhat[..., :4])


def test_backward_workspace_is_bounded():
    """The sorted backward's workspace: 16 bytes a slot and the counts of at most 256 chunks of queries, for what is
    sorted at a time -- at most 2^26 slots, or one query's."""
    from treeattn_amd import _lib
    size = _lib.lib().ta_sparse_attn_bwd_workspace_size
    counts = (2048 * 256 + 2) * 4   # and a word to align what comes in pairs
    for B, H, T, KC in [(1, 1, 1, 1), (2, 6, 4096, 52), (1, 1, 262144, 52), (1, 1, 16384, 2100), (1, 3, 300, 5000)]:
        assert 0 < size(B, H, T, KC) - 16 * B * H * T * KC <= B * H * counts, (B, H, T, KC)
    for B, H, T, KC in [(4096, 12, 256, 52), (1, 16, 16384, 2100), (65535, 1, 16, 16), (1, 1, (1 << 22) + 5, 600)]:
        assert size(B, H, T, KC) <= (1 << 30) + counts, (B, H, T, KC)
    assert size(1, 1, 3, 1 << 27) <= (16 << 27) + counts
    assert size(0, 1, 8, 8) == size(1, 1, 0, 8) == size(1, 1, 8, 0) == 0


def test_backward_route_choice():
    """The default dk/dv route: the fixed (bit-reproducible) order up to SORTED_MAX_POSITIONS queries and keys, the atomic
    adds past it, whatever the number of pairs and slots (the workspace is bounded)."""
    from treeattn_amd import kernels as K
    most = K.SORTED_MAX_POSITIONS
    assert K.sorted_by_default(512, 512) and K.sorted_by_default(32768, 32768) and K.sorted_by_default(most, most)
    assert not K.sorted_by_default(most + 1, 64) and not K.sorted_by_default(64, most + 1)


def test_tracing_builds_are_separate():
    """The phase marks are nothing in the library build: it exports no trace buffer accessor, and a tracing build
    of one source lives in its own library beside it."""
    from treeattn_amd import _lib, build, phase_trace  # noqa: F401
    L = _lib.lib()
    assert not hasattr(L, 'ta_trace_read')
    assert build.trace_lib_path('attend.hip') != _lib.LIB_PATH
    assert build.trace_lib_path('attend.hip').endswith('libtreeattn_trace_attend.so')
