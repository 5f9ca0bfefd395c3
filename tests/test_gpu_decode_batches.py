"""int8 and int4 matmuls of up to 16 rows: on the narrow tiles, where those are estimated to be ahead of the bandwidth-bound kernels, and on what is ahead of them (strips on
small weights). Exact on small integers, with part of a row block, a bias, strides, K in pieces and whole; the workspace is zero where it has to be; equal to what a captured graph
computes; a wanted number of K parts still goes to the bandwidth-bound kernel."""
import numpy as np
import pytest
import torch

from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, last_launch

pytestmark = pytest.mark.gpu


def _int8(m, k, n, seed=0):
    rng = np.random.default_rng(m * 7 + k + n + seed)
    a, q = rng.integers(-3, 4, (m, k)).astype(np.float16), rng.integers(-2, 3, (k, n)).astype(np.int8)
    exact = a.astype(np.float32) @ q.astype(np.float32)
    assert np.abs(exact).max() <= 2048  # (exact in float16)
    return dev(a), dev(q), torch.from_numpy(exact)


@pytest.mark.parametrize('m', [1, 4, 8, 9, 15, 16])
@pytest.mark.parametrize('k,n', [(768, 132), (1000, 2048), (1024, 8192), (2048, 2500), (4096, 4096), (9152, 2640)])
def test_int8(m, k, n):
    announce('int8 decode batch', m, k, n)
    a, q, exact = _int8(m, k, n)
    one = torch.ones(n, dtype=torch.float16, device='cuda')
    assert torch.equal(quant.symmetric_quant_matmul(a, q, one).float().cpu(), exact)
    bias = (torch.arange(n, device='cuda') % 5).half()
    assert torch.equal(quant.symmetric_quant_matmul(a, q, one, bias).float().cpu(), (exact.half() + bias.cpu()).float())
    assert not ffi.workspace(a.device)[:65536 + (16 << 20)].any()


@pytest.mark.parametrize('dtype', ['bfloat16', 'float16'])
@pytest.mark.parametrize('m', [1, 5, 16])
@pytest.mark.parametrize('k,n,group', [(768, 136, 64), (1024, 4096, 128), (2048, 2504, 128), (1152, 4360, 128), (4096, 4096, 128), (6144, 1024, 64), (960, 520, 96)])
def test_int4(m, k, n, group, dtype):
    announce('int4 decode batch', m, k, n, group, dtype)
    rng = np.random.default_rng(m + k + n)
    a, q = rng.integers(-1, 2, (m, k)).astype(np.float32), rng.integers(-7, 8, (k, n))
    packed = dev(((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).astype(np.uint8))
    scales = 2.0 ** rng.integers(-2, 1, (k // group, n)).astype(np.float32)
    exact = torch.from_numpy(a @ (q * np.repeat(scales, group, axis=0)).astype(np.float32))
    ty = getattr(torch, dtype)
    got = quant.symmetric_quant_matmul_w4a16(dev(a).to(ty), packed, dev(scales).to(ty), group)
    assert torch.equal(got.cpu(), exact.to(ty))


# sizes that the kernels of strips leave to the narrow tiles
@pytest.mark.parametrize('m', [9, 15, 16])
@pytest.mark.parametrize('k,n', [(2624, 132), (2880, 1000), (3002, 2500), (4096, 2048), (9152, 2640)])
def test_int8_on_the_narrow_tiles(m, k, n):
    announce('int8 decode batch on the narrow tiles', m, k, n)
    a, q, exact = _int8(m, k, n, 1)
    assert torch.equal(quant.symmetric_quant_matmul(a, q, torch.ones(n, dtype=torch.float16, device='cuda')).float().cpu(), exact)
    assert 'gemm_mid_kernel' in last_launch()[0]
    assert not ffi.workspace(a.device)[:65536 + (16 << 20)].any()


@pytest.mark.parametrize('k,n,group', [(3072, 520, 128), (4096, 4096, 128), (6144, 1024, 64), (3840, 2504, 128)])
def test_int4_on_the_narrow_tiles(k, n, group):
    announce('int4 decode batch on the narrow tiles', k, n, group)
    rng = np.random.default_rng(k + n)
    a, q = rng.integers(-1, 2, (16, k)).astype(np.float32), rng.integers(-7, 8, (k, n))
    packed = dev(((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).astype(np.uint8))
    scales = 2.0 ** rng.integers(-2, 1, (k // group, n)).astype(np.float32)
    exact = torch.from_numpy(a @ (q * np.repeat(scales, group, axis=0)).astype(np.float32))
    got = quant.symmetric_quant_matmul_w4a16(dev(a).bfloat16(), packed, dev(scales).bfloat16(), group)
    assert 'gemm_mid_kernel' in last_launch()[0]
    assert torch.equal(got.cpu(), exact.bfloat16())


def test_wanted_parts_and_strides():
    announce('int8 decode batch: parts, strides')
    a, q, exact = _int8(16, 2048, 2048)
    one = torch.ones(2048, dtype=torch.float16, device='cuda')
    ws = ffi.workspace(a.device)
    for parts in (0, 1, 4):
        c = torch.empty((16, 2048), dtype=torch.float16, device='cuda')
        ffi.call('hidet_symmetric_quant_matmul_f16_i8', a, q, one, c, 16, 2048, 2048, 2048, parts, ws, ws.numel(), ffi.current_stream(a.device))
        assert torch.equal(c.float().cpu(), exact)
    wide = torch.zeros((16, 2050), dtype=torch.float16, device='cuda')
    wide[:, :2048] = a
    assert torch.equal(quant.symmetric_quant_matmul(wide[:, :2048], q, one).float().cpu(), exact)


def test_replayed_graph():
    announce('int8 decode batch: graph')
    a, q, exact = _int8(8, 4096, 2048)
    one = torch.ones(2048, dtype=torch.float16, device='cuda')
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        quant.symmetric_quant_matmul(a, q, one)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = quant.symmetric_quant_matmul(a, q, one)
    for i in range(4):
        got.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got.float().cpu(), exact)
        assert 'gemm_mid_kernel' in last_launch()[0]
        quant.symmetric_quant_matmul(a, q, one)
