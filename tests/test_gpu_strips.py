"""The kernels of strips of columns over all of K, every variant by its name (the operators choose by estimated times, which leaves some of them to sizes that no
list of shapes is sure to contain): row blocks, columns, waves, two row tiles and part of a third, N that ends inside a strip, waves without a step of K, K that ends inside a
step. Small integers whose results the output type holds must be equal; ordinary values stay within the rounding of float32 sums and of the result."""
import numpy as np
import pytest
import torch

from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, last_launch, variant
from test_gpu_fp8_tiles import operands

pytestmark = pytest.mark.gpu

ROW_BLOCKS = [1, 2, 3, 4]


def _stream():
    return ffi.current_stream(torch.device('cuda'))


def _launched(kernel, *arguments):
    assert variant(kernel, *arguments) in last_launch()[0], last_launch()


def _int8(m, k, n):
    rng = np.random.default_rng(m + k + n)
    a, q = rng.integers(-2, 3, (m, k)).astype(np.float16), rng.integers(-2, 3, (k, n)).astype(np.int8)
    a *= rng.random((m, k)) < 0.5
    q[0, 0], q[k - 1, n - 1] = 127, -128
    exact = a.astype(np.float32) @ q.astype(np.float32)
    assert np.abs(exact).max() <= 2048
    return dev(a), dev(q), torch.from_numpy(exact)


@pytest.mark.parametrize('k,n', [(128, 6), (1152, 74), (130, 4), (1118, 130)])
@pytest.mark.parametrize('columns', [2, 4])
@pytest.mark.parametrize('rows', ROW_BLOCKS)
def test_int8(rows, columns, k, n):
    announce('strips int8', rows, columns, k, n)
    m = 32 * rows + 5
    a, q, exact = _int8(m, k, n)
    one, bias, c = torch.ones(n, dtype=torch.float16, device='cuda'), (torch.arange(n, device='cuda') % 7).half(), torch.full((m, n), float('nan'), dtype=torch.float16, device='cuda')
    ffi.call('hidet_qmm_strips_f16_i8', rows, columns, a, q, one, bias, c, m, k, n, k, _stream())
    _launched('skinny_w8a16_small_kernel', k % 128 != 0, rows, columns)
    assert torch.equal(c.cpu(), exact.half() + bias.cpu())


@pytest.mark.parametrize('k,n', [(16, 5), (1152, 67), (1040, 40)])
@pytest.mark.parametrize('groups', [1, 2])
@pytest.mark.parametrize('rows', ROW_BLOCKS)
def test_int8_k_contiguous(rows, groups, k, n):
    announce('strips int8 K-contiguous', rows, groups, k, n)
    m = 32 * rows + 5
    a, q, exact = _int8(m, k, n)
    one, c = torch.ones(n, dtype=torch.float16, device='cuda'), torch.full((m, n), float('nan'), dtype=torch.float16, device='cuda')
    ffi.call('hidet_qmm_strips_f16_i8_nk', rows, groups, a, q.T.contiguous(), one, None, c, m, k, n, k, k, _stream())
    _launched('skinny_w8a16_nk_tall_kernel', k % 128 != 0, rows, groups)
    assert torch.equal(c.cpu(), exact.half())


@pytest.mark.parametrize('dtype', ['bfloat16', 'float16'])
@pytest.mark.parametrize('k,n,group', [(128, 8, 64), (1152, 136, 128), (2304, 40, 256)])
@pytest.mark.parametrize('columns,waves', [(2, 8), (4, 8), (2, 16)])
@pytest.mark.parametrize('rows', ROW_BLOCKS)
def test_int4(rows, columns, waves, k, n, group, dtype):
    if waves == 16 and rows > 1:
        return
    announce('strips int4', rows, columns, waves, k, n, group, dtype)
    m, ty = 32 * rows + 5, getattr(torch, dtype)
    rng = np.random.default_rng(m + k + n)
    a, q = rng.integers(-1, 2, (m, k)).astype(np.float32), rng.integers(-8, 8, (k, n))
    scales = 2.0 ** rng.integers(-2, 1, (k // group, n)).astype(np.float32)
    exact = torch.from_numpy(a @ (q * np.repeat(scales, group, axis=0)).astype(np.float32))
    packed = dev(((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).astype(np.uint8))
    c = torch.full((m, n), float('nan'), dtype=ty, device='cuda')
    ffi.call('hidet_qmm_strips_w4a16', rows, columns, waves, dev(a).to(ty), packed, dev(scales).to(ty), None, c, m, k, n, k, group, ffi.DTYPE_CODE[ty], _stream())
    _launched('skinny_w4a16_small_kernel', ffi.DTYPE_CODE[ty], 4 if group % 128 == 0 else 2, waves, rows, columns)
    assert torch.equal(c.cpu(), exact.to(ty))


@pytest.mark.parametrize('k,n,scaled', [(16, 5, False), (1152, 67, False), (1136, 40, False), (128, 128, True), (1152, 256, True)])
@pytest.mark.parametrize('groups', [1, 2])
@pytest.mark.parametrize('rows', ROW_BLOCKS)
def test_fp8(rows, groups, k, n, scaled):
    announce('strips fp8', rows, groups, k, n, scaled)
    m = 32 * rows + 5
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, False)
    c = torch.full((m, n), float('nan'), dtype=torch.float32, device='cuda')
    if scaled:
        sa, sb = rng.integers(1, 5, (k // 128, m)).astype(np.float32), rng.integers(1, 5, (n // 128, k // 128)).astype(np.float32)
        exact = (ai * np.repeat(sa.T, 128, axis=1)).astype(np.float64) @ (bi * np.repeat(np.repeat(sb, 128, axis=0), 128, axis=1)).T.astype(np.float64)
        scales = dev(sa), dev(sb)
    else:
        exact, scales = ai.astype(np.float64) @ bi.T * 0.5, (torch.full((), 0.5, device='cuda'), None)
    assert np.abs(exact).max() < 2 ** 24
    ffi.call('hidet_qmm_strips_f8', rows, groups, int(scaled), a, b, c, m, n, k, k, k, ffi.F32, *scales, _stream())
    _launched('skinny_fp8_tall_kernel', scaled, k % 128 != 0, rows, groups)
    assert np.array_equal(c.cpu().numpy(), exact.astype(np.float32))


# Through the operators, values and scales as a program has them. float32 sums of k products by steps of `deep` of them: each adds an error of at most 2^-24 of the magnitudes summed so
# far per addition, whatever the order inside a step; then half a unit of the result (two where a group's scale or a code's rounding comes before).
def _close(got, want, magnitudes, additions, unit):
    bound = magnitudes * 2.0 ** -24 * additions + want.abs() * unit + 2.0 ** -24
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize('m,k,n', [(7, 1024, 2050), (40, 1090, 1500), (100, 512, 3000)])
def test_int8_ordinary_values(m, k, n):
    announce('strips int8: ordinary values', m, k, n)
    g = torch.Generator(device='cuda').manual_seed(m)
    w, scale = quant.symmetric_quantize(torch.randn((k, n), generator=g, device='cuda') * 0.02, 'int8', dims=0)
    x, scale = torch.randn((m, k), generator=g, device='cuda').half(), scale.half()
    got = quant.symmetric_quant_matmul(x, w, scale)
    assert 'skinny_w8a16_small_kernel' in last_launch()[0]
    _close(got, (x.double() @ w.double()) * scale.double(), (x.double().abs() @ w.double().abs()) * scale.double(), k, 2.0 ** -11)


@pytest.mark.parametrize('dtype', ['bfloat16', 'float16'])
@pytest.mark.parametrize('m,k,n,group', [(5, 1024, 2048, 128), (40, 1536, 3072, 64)])
def test_int4_ordinary_values(m, k, n, group, dtype):
    announce('strips int4: ordinary values', m, k, n, group, dtype)
    ty = getattr(torch, dtype)
    g = torch.Generator(device='cuda').manual_seed(m)
    packed, scales = quant.symmetric_group_quantize_int4(torch.randn((k, n), generator=g, device='cuda') * 0.02, group, ty)
    x = torch.randn((m, k), generator=g, device='cuda').to(ty)
    got = quant.symmetric_quant_matmul_w4a16(x, packed, scales, group)
    assert 'skinny_w4a16_small_kernel' in last_launch()[0]
    p = packed.to(torch.int32)
    q = torch.stack([p & 15, p >> 4], dim=2).reshape(k, n)
    w = (q - 16 * (q > 7)).double() * scales.double().repeat_interleave(group, dim=0)
    _close(got, x.double() @ w, x.double().abs() @ w.abs(), k, 2.0 ** -8 if dtype == 'bfloat16' else 2.0 ** -11)


@pytest.mark.parametrize('scaled', [False, True])
@pytest.mark.parametrize('m,k,n', [(24, 1024, 2048), (50, 2048, 1024)])
def test_fp8_ordinary_values(m, k, n, scaled):
    from hidet_amd.graph.ops.matmul import matmul_f8 as F8

    announce('strips fp8: ordinary values', m, k, n, scaled)
    g = torch.Generator(device='cuda').manual_seed(m)
    a = (torch.randn((m, k), generator=g, device='cuda') * 150).clamp(-448, 448).to(torch.float8_e4m3fn)
    b = (torch.randn((n, k), generator=g, device='cuda') * 110).clamp(-448, 448).to(torch.float8_e4m3fn)
    if scaled:
        sa, sb = torch.rand((k // 128, m), generator=g, device='cuda') / 448 + 0.005, torch.rand((n // 128, k // 128), generator=g, device='cuda') / 448 + 0.008
        got = F8.matmul_f8_scaled(a, b, sa, sb, output_dtype='float32')
        ad, bd = a.double() * sa.double().T.repeat_interleave(128, dim=1), b.double() * sb.double().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)
    else:
        sa, sb = torch.full((), 0.007, device='cuda'), torch.full((), 0.0003, device='cuda')
        got = F8.matmul_f8_per_tensor(a, b, sa, sb, output_dtype=torch.float32)
        ad, bd = a.double() * sa.double(), b.double() * sb.double()
    assert 'skinny_fp8_tall_kernel' in last_launch()[0]
    _close(got, ad @ bd.T.contiguous(), ad.abs() @ bd.abs().T.contiguous(), k, 2.0 ** -22)
