"""int4 matmuls on small weights, which one workgroup per column strip computes over all of K: several row tiles, waves without a
step of K, groups of 64, 128 and more, columns past the end, a bias, strides; and sizes next to those that take this kernel
(its variants by name: test_gpu_strips.py). Small integers and scales of powers of
two: the results must be equal."""
import numpy as np
import pytest
import torch

from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, last_launch

pytestmark = pytest.mark.gpu


def _case(m, k, n, group, dtype):
    rng = np.random.default_rng(m + k + n + group)
    a, q = rng.integers(-1, 2, (m, k)).astype(np.float32), rng.integers(-8, 8, (k, n))
    scales = 2.0 ** rng.integers(-2, 1, (k // group, n)).astype(np.float32)
    exact = torch.from_numpy(a @ (q * np.repeat(scales, group, axis=0)).astype(np.float32))
    packed = dev(((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).astype(np.uint8))
    return dev(a).to(dtype), packed, dev(scales).to(dtype), exact


@pytest.mark.parametrize('dtype', ['bfloat16', 'float16'])
@pytest.mark.parametrize('m', [1, 16, 17, 33, 49, 64, 65, 130, 300])
@pytest.mark.parametrize('k,n,group', [(128, 8, 128), (128, 40, 64), (384, 264, 128), (1024, 64, 256), (1024, 3000, 128), (1152, 2056, 64), (2048, 2048, 128), (2048, 6144, 128), (2176, 1024, 64), (2944, 136, 128), (3072, 2048, 64), (3200, 520, 128), (4096, 520, 256), (4224, 264, 128)])
def test_exact(m, k, n, group, dtype):
    announce('int4 small weight', m, k, n, group, dtype)
    ty = getattr(torch, dtype)
    a, packed, scales, exact = _case(m, k, n, group, ty)
    got = quant.symmetric_quant_matmul_w4a16(a, packed, scales, group)
    assert torch.equal(got.cpu(), exact.to(ty))


def test_bias_and_strides():
    announce('int4 small weight: bias, strides')
    m, k, n, group = 20, 512, 264, 128
    a, packed, scales, exact = _case(m, k, n, group, torch.bfloat16)
    wide = torch.zeros((m, k + 2), dtype=torch.bfloat16, device='cuda')
    wide[:, :k] = a
    bias = (torch.arange(n, device='cuda') % 5).bfloat16()
    ws = ffi.workspace(a.device)
    c = torch.empty((m, n), dtype=torch.bfloat16, device='cuda')
    ffi.call('hidet_symmetric_quant_matmul_w4a16_bias', wide, packed, scales, bias, c, m, k, n, k + 2, group, ffi.DTYPE_CODE[torch.bfloat16], 0, ws, ws.numel(), ffi.current_stream(a.device))
    assert torch.equal(c.cpu(), exact.bfloat16() + bias.cpu())


@pytest.mark.parametrize('m,k,n,strips', [(504, 1024, 7040, False), (150, 1024, 11008, False), (64, 1024, 4096, True)])
def test_strips_of_up_to_two_rounds_of_the_chip(m, k, n, strips):
    announce('int4 small weight: rounds', m, k, n)
    a, packed, scales, exact = _case(m, k, n, 128, torch.bfloat16)
    got = quant.symmetric_quant_matmul_w4a16(a, packed, scales, 128)
    assert ('skinny_w4a16_small' in last_launch()[0]) == strips
    assert torch.equal(got.cpu(), exact.bfloat16())
