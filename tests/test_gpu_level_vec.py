"""Level sums: the pass of 16-byte slices against the element pass (which rows off 16-byte alignment take), bit for bit,
around whole segments of 16 and 64 rows and whole chunks, over one and two passes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda'


@pytest.mark.parametrize('dtype,D', [(torch.float32, 16), (torch.float32, 128), (torch.float16, 64), (torch.bfloat16, 32),
                                     (torch.bfloat16, 128)])
@pytest.mark.parametrize('t_end', [1, 15, 16, 17, 255, 1023, 1024, 2049, 8191, 8192])
def test_level_vec_equals_element_pass(dtype, D, t_end):
    from treeattn_amd import kernels as K
    B, H, T = 1, 2, 8192
    g = torch.Generator().manual_seed(t_end)
    k = torch.randn(B, H, T, D, generator=g).to(dtype).to(DEV)
    off = torch.empty(k.numel() + 1, dtype=dtype, device=DEV)[1:].view_as(k).copy_(k)
    assert off.data_ptr() % 16
    shape = K.TreeShape(T, 2, 2)
    for i, (a, b) in enumerate(zip(K.level_sums(k, shape.blevels, t_end=t_end), K.level_sums(off, shape.blevels, t_end=t_end))):
        n = t_end >> shape.blevels[i]   # complete nodes
        assert torch.equal(a[:, :, :n], b[:, :, :n]), shape.blevels[i]


@pytest.mark.parametrize('B,T,D,dtype', [
    (65, 4096, 64, torch.bfloat16),    # more than 1024 workgroups of whole chunks: segments of 64 rows
    (64, 4096, 64, torch.bfloat16),    # 1024 of them: segments of 16
    (33, 4095, 64, torch.float16),     # ragged chunks, past 256 workgroups
    (33, 1025, 128, torch.float32),    # a chunk of one row
    (40, 8256, 32, torch.float16),     # chunks of 4096 rows, the last of one segment
])
def test_many_workgroups_equal_element_pass(B, T, D, dtype):
    from treeattn_amd import kernels as K
    H = 8
    g = torch.Generator(device=DEV).manual_seed(T)
    k = torch.randn(B, H, T, D, generator=g, device=DEV).to(dtype)
    off = torch.empty(k.numel() + 1, dtype=dtype, device=DEV)[1:].view_as(k).copy_(k)
    blevels = list(range(1, T.bit_length()))
    for l, a, b in zip(blevels, K.level_sums(k, blevels), K.level_sums(off, blevels)):
        assert torch.equal(a, b), l
