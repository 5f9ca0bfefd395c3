"""NaN, infinities and values near the ends of the types' ranges, where a kernel's shortcut can differ from its definition."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from hidet_amd.graph.ops.matmul import matmul_f8 as F8
from gpu_util import announce, dev

pytestmark = pytest.mark.gpu


# one launch and two, sizes of whole quads and not, tensors that start off their quads; next to a NaN both the product with the
# reciprocal and the division (a value on a tie of the format) have to leave it alone
@pytest.mark.parametrize('numel', [4, 1027, 4096, 65536, 70001, 1 << 17])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('offset', [0, 1])
def test_fp8_quantization_keeps_nan(numel, dtype, offset):
    announce('fp8 nan', numel, dtype, offset)
    rng = np.random.default_rng(numel)
    x = rng.standard_normal(numel + offset).astype(np.float32)
    x[offset] = 448.0  # the scale is one: 1.0625 and 2.125 lie on ties, and so does the largest value on its boundary
    x[offset + 2::7] = np.nan
    x[offset + 3::11] = -np.nan
    x[offset + 3:offset + 20:4] = 1.0625
    x = np.clip(x, -448, 448)
    t = dev(x).to(dtype)[offset:]
    codes, scale = F8.fp8_quantize_per_tensor(t)
    assert scale.item() == 1.0
    assert np.array_equal(codes.view(torch.uint8).cpu().numpy(), O.e4m3_encode(t.float().cpu().numpy()))


def test_fp8_quantization_of_infinities_and_subnormal_scales():
    announce('fp8 inf')
    x = torch.tensor([float('inf'), 3.0, -2.0, 0.0, float('-inf')], device='cuda')
    codes, scale = F8.fp8_quantize_per_tensor(x)
    c = codes.view(torch.uint8).cpu().numpy()
    assert np.isinf(scale.item()) and list(c[1:4] & 0x7F) == [0, 0, 0] and list(c[[0, 4]] & 0x7F) == [0x7F, 0x7F]  # inf / inf
    tiny = np.array([700, -700, 350, 1], np.float32) * np.float32(2.0 ** -149)  # the scale is two of the smallest units
    codes, scale = F8.fp8_quantize_per_tensor(dev(tiny))
    c0, s0 = O.fp8_quantize_per_tensor(tiny)
    assert np.float32(scale.item()) == s0 and np.array_equal(codes.view(torch.uint8).cpu().numpy(), c0)


# an odd number of k blocks: a group of waves has a stage past the end in its last round; one and several pieces of K
@pytest.mark.parametrize('m,k,n', [(17, 128, 128), (40, 384, 256), (64, 7040, 384), (130, 1152, 512)])
def test_block_scaled_fp8_with_infinite_scales(m, k, n):
    announce('fp8 block scales inf', m, k, n)
    g = torch.Generator(device='cuda').manual_seed(m + k)
    a = torch.randint(1, 4, (m, k), generator=g, device='cuda').float()
    a[::3] *= -1
    b = torch.randint(1, 4, (n, k), generator=g, device='cuda').float()
    scale_a, scale_b = torch.full((k // 128, m), 0.5, device='cuda'), torch.full((n // 128, k // 128), 0.25, device='cuda')
    scale_b[0, 0] = float('inf')
    scale_a[-1, 5] = float('inf')
    part = torch.matmul(a.view(m, k // 128, 128).transpose(0, 1).double().contiguous(), b.view(n, k // 128, 128).permute(1, 2, 0).double().contiguous())
    want = (part * scale_a.double()[:, :, None] * scale_b.double().repeat_interleave(128, 0).t()[:, None, :]).sum(0).float()
    assert not want.isnan().any() and want.isinf().any()
    for _ in range(2):
        assert torch.equal(F8.matmul_f8_scaled(a.to(F8.f8e4m3), b.to(F8.f8e4m3), scale_a, scale_b, output_dtype='float32'), want)
