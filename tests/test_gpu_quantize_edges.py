"""The quantizers at the edges of their kernels' tiles, on values at and next to the rounding ties of a scale that is no
power of two (where a product with the scale's reciprocal and the quotient could round apart): bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from hidet_amd.graph.ops.matmul import matmul_f8 as F8
from gpu_util import announce, dev, fastest_ms, host

pytestmark = pytest.mark.gpu


def _near_ties(rng, shape, axis, qmax):
    """Normal values, half of them replaced by (n + 1/2) * scale of their slice and its two float32 neighbours."""
    w = (rng.standard_normal(shape) * 0.02).astype(np.float32)
    s = (np.abs(w).max(axis=axis, keepdims=True) / np.float32(qmax)).astype(np.float32)
    tie = ((np.floor(w / s).clip(-qmax, qmax - 1) + np.float32(0.5)) * s).astype(np.float32)
    pick = rng.integers(0, 8, shape)
    w = np.where(pick == 0, tie, w)
    w = np.where(pick == 1, np.nextafter(tie, np.float32(1)), w)
    return np.where(pick == 2, np.nextafter(tie, np.float32(-1)), w).astype(np.float32)


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('shape,dim,codes', [((1, 3), 0, 'int8'), ((63, 255), 0, 'int8'), ((65, 257), 0, 'int16'), ((4100, 1026), 0, 'int8'),
                                             ((129, 6), 0, 'int8'), ((3, 2049, 130), 1, 'int8'), ((33, 16387), 1, 'int8'), ((5, 4100), 1, 'int16'),
                                             ((520, 66, 9), 1, 'int8'), ((521, 3, 7), 1, 'int16'), ((9, 130, 63), 1, 'int8'), ((513, 5, 64), 1, 'int8'), ((513, 300, 2), 1, 'int8'), ((3, 4096), 1, 'int8'), ((3, 8192), 1, 'int16'), ((3, 8196), 1, 'int8'), ((2, 16384), 1, 'int8'), ((2, 16388), 1, 'int8'),
                                             # 2, 4 and 8 rows per thread: the last matrices of one form and the first of the next
                                             ((17, 1026), 0, 'int8'), ((8192, 256), 0, 'int8'), ((8193, 256), 0, 'int16'), ((1025, 6144), 0, 'int8'), ((1024, 6146), 0, 'int8'), ((2, 65, 514), 1, 'int8'), ((3, 2100, 95), 1, 'int8'), ((600, 9, 96), 1, 'int8'),
                                             # tall: many row ranges, whose maxima one more launch puts together
                                             ((50001, 9), 0, 'int8'), ((2, 30000, 3), 1, 'int16'), ((20000, 95), 0, 'int8'), ((70001, 66), 0, 'int8'), ((70000, 130), 0, 'int8'),
                                             ((2, 20000, 260), 1, 'int8'), ((2, 66000, 96), 1, 'int8')])
def test_columns_and_rows_bit_exact(shape, dim, codes, dtype):
    announce('quantize edges', shape, dim, codes, dtype)
    w = _near_ties(np.random.default_rng(shape[-1]), shape, dim, 127 if codes == 'int8' else 32767)
    w.reshape(-1, shape[-1])[:, 0] = 0  # a column of zeros
    if dtype == 'bfloat16':
        w = O.to_bf16(w)
    elif dtype == 'float16':
        w = w.astype(np.float16)
    q0, s0 = O.symmetric_quantize(w, codes, dim, dtype=dtype, target='cpu' if dtype == 'float32' else 'gpu')
    q, s = quant.symmetric_quantize(dev(w).to(getattr(torch, dtype)), codes, dim)
    assert np.array_equal(host(q), q0)
    assert np.array_equal(s.float().cpu().numpy(), np.asarray(s0, dtype=np.float32))
    assert np.array_equal(quant.symmetric_dequantize(q, s, dim).float().cpu().numpy(),
                          np.asarray(O.symmetric_dequantize(q0, s0, dim, dtype=dtype), dtype=np.float32))


# more slices than a grid has layers
@pytest.mark.parametrize('shape', [(65536, 3, 5), (65537, 2, 64)])
def test_dequantize_of_many_slices(shape):
    announce('dequantize of many slices', shape)
    rng = np.random.default_rng(shape[2])
    q = rng.integers(-127, 128, shape).astype(np.int8)
    s = rng.random((shape[0], shape[2])).astype(np.float32)
    got = quant.symmetric_dequantize(dev(q), dev(s), 1).cpu().numpy()
    assert np.array_equal(got, q.astype(np.float32) * s[:, None, :])


# the same for the quantizer, whose slices then take several launches, and rows of more than one launch's threads
@pytest.mark.parametrize('shape', [(65535, 3, 5), (65536, 3, 5), (131071, 2, 9), (65537, 2, 100), (262144, 6), (262145, 7), ((1 << 24) + 3, 4)])
def test_quantize_of_many_slices(shape):
    announce('quantize of many slices', shape)
    w = torch.randn(shape, generator=torch.Generator(device='cuda').manual_seed(shape[0]), device='cuda')
    q, s = quant.symmetric_quantize(w, 'int8', 1)
    for part in (slice(0, 1000), slice(65000, 66000), slice(shape[0] - 1000, shape[0])):
        q0, s0 = O.symmetric_quantize(host(w[part]), 'int8', 1)
        assert np.array_equal(host(q[part]), q0) and np.array_equal(host(s[part]), s0)
    assert torch.equal(s, w.abs().amax(1) / torch.full_like(s, 127))  # (by a number torch multiplies with its reciprocal)


def test_more_scales_than_the_standing_workspace_holds():
    announce('quantize with 22 million scales')
    w = torch.randn((2, 22_000_000), device='cuda')
    q, s = quant.symmetric_quantize(w, 'int8', 0)
    assert torch.equal(s, w.abs().amax(0) / torch.full_like(s, 127))
    for part in (slice(0, 1000), slice(-1000, None)):
        assert np.array_equal(host(q[:, part]), O.symmetric_quantize(host(w[:, part]), 'int8', 0)[0])


@pytest.mark.parametrize('k,n,group', [(4, 2, 4), (96, 258, 32), (66, 254, 33), (128, 1030, 64), (256, 126, 128), (390, 130, 65), (512, 66, 256),
                                       (514, 6, 257), (1024, 258, 1024)])
def test_int4_groups_bit_exact(k, n, group):
    announce('int4 edges', k, n, group)
    w = _near_ties(np.random.default_rng(k + n), (k // group, group, n), 1, 7).reshape(k, n)
    packed, scales = quant.symmetric_group_quantize_int4(dev(w), group, 'float16')
    p0, s0, _ = O.group_quantize_int4(w, group, 'float16')
    assert np.array_equal(host(packed), p0) and np.array_equal(host(scales).view(np.uint16), s0.view(np.uint16))


@pytest.mark.parametrize('numel', [65535, 65537, 8 * 4096 - 4, 4096 * 1024 * 2 + 3])
def test_fp8_per_tensor_bit_exact(numel):
    announce('fp8 edges', numel)
    rng = np.random.default_rng(numel)
    x = (rng.standard_normal(numel) * 3).astype(np.float32)
    vals = O.e4m3_decode(np.arange(0, 0x7F, dtype=np.uint8)).astype(np.float64)
    ties = ((vals[:-1] + vals[1:]) / 2 * (float(np.abs(x).max()) / 448)).astype(np.float32)
    ties = np.concatenate([ties, np.nextafter(ties, np.float32(0)), np.nextafter(ties, np.float32(9)), np.zeros(5, np.float32)])
    x[rng.permutation(numel)[:ties.size]] = ties
    for t in (dev(x), dev(x).bfloat16(), dev(x).half()):
        codes, scale = F8.fp8_quantize_per_tensor(t)
        c0, s0 = O.fp8_quantize_per_tensor(t.float().cpu().numpy())
        assert np.float32(scale.item()) == s0 and np.array_equal(codes.view(torch.uint8).cpu().numpy(), c0)


# one value, around a workgroup's 4096 elements, the last size of the single launch and the first behind it; the largest value
# at the end, where only the last workgroup converts it
@pytest.mark.parametrize('numel', [4, 4092, 4096, 4100, 20000, 65536, 65540])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_fp8_per_tensor_of_a_few_rows(numel, dtype):
    announce('fp8 few rows', numel, dtype)
    x = np.random.default_rng(numel).standard_normal(numel).astype(np.float32)
    x[-1] = 9.0
    t = dev(x).to(dtype)
    codes, scale = F8.fp8_quantize_per_tensor(t)
    c0, s0 = O.fp8_quantize_per_tensor(t.float().cpu().numpy())
    assert np.array_equal(codes.view(torch.uint8).cpu().numpy(), c0)
    assert scale.item() == float(np.asarray(s0).reshape(-1)[0])


# 16-bit inputs whose quotients are often rounding boundaries of the format (448 or 3/4 of it, by powers of two) or one float32 away
# from one; the largest sizes of one launch and of one vector per thread, and the first behind them
@pytest.mark.parametrize('numel', [65536, 65544, 2048 * 2048, 2048 * 2048 + 8])
@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_fp8_per_tensor_of_ties(numel, dtype):
    announce('fp8 ties', numel, dtype)
    rng = np.random.default_rng(numel)
    for amax in (5.125, 3.5, 7.9375, 1.0):
        x = amax * np.exp2(-rng.integers(0, 19, numel)) * rng.choice([1, 3 / 4, 1 / 2, 17 / 28, 5 / 7, 25 / 28, 31 / 32, 0.9], numel)
        x = (x * rng.choice([-1, 1], numel)).astype(np.float32)
        x[numel // 2] = amax
        t = dev(x).to(dtype)
        codes, scale = F8.fp8_quantize_per_tensor(t)
        c0, s0 = O.fp8_quantize_per_tensor(t.float().cpu().numpy())
        assert np.float32(scale.item()) == s0 and np.array_equal(codes.view(torch.uint8).cpu().numpy(), c0)


# an empty reduction: scales of zero, and nothing behind the last of them (a number of 16-bit scales that fills no whole word)
@pytest.mark.parametrize('count', [1, 3, 256, 257])
@pytest.mark.parametrize('start', [0, 1])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
def test_scales_of_an_empty_reduction(count, start, dtype):
    announce('empty reduction', count, start, dtype)
    buf = torch.full((count + 4,), 7.0, dtype=dtype, device='cuda')
    scale = buf[start:start + count]
    ws = ffi.workspace(buf.device)
    none = torch.empty((0,), dtype=torch.int8, device='cuda')
    ffi.call('hidet_symmetric_quantize', none, none, scale, 1, 0, count, ffi.DTYPE_CODE[dtype], ffi.DTYPE_CODE[torch.int8], ws, ws.numel(),
             ffi.current_stream(buf.device))
    want = torch.full_like(buf, 7.0)
    want[start:start + count] = 0
    assert torch.equal(buf, want)


@pytest.mark.parametrize('inner', [9, 64, 128])
def test_tall_weights_cost_no_more_than_others(inner):
    """Maxima over a long axis of a few columns keep the whole chip at work (32 workgroups took ten times as long)."""
    announce('quantize tall', inner)
    rows = (1 << 24) // inner
    tall, square = torch.randn((rows, inner), device='cuda'), torch.randn((4096, 4096), device='cuda')
    assert fastest_ms(lambda: quant.symmetric_quantize(tall, 'int8', 0)) < 3 * fastest_ms(lambda: quant.symmetric_quantize(square, 'int8', 0))
