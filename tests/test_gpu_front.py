"""The native front of the operators: what it handles equals the Python path bit for bit, and what it does not handle (it
returns None) still works or raises as before."""
import pytest
import torch

from hidet_amd import BackendException, ffi
from hidet_amd.graph.ops import quant
from hidet_amd.graph.ops.matmul import matmul_f8 as F8
from hidet_amd.graph.ops.quant import group_int4, symmetric
from hidet_amd.graph.ops.quant.matmul import run_w8a16
from hidet_amd.graph.ops.quant.group_int4 import _run_w4a16
from gpu_util import announce

pytestmark = pytest.mark.gpu


def _case(m, k, n):
    g = torch.Generator(device='cuda').manual_seed(m + k + n)
    x = torch.randn((m, k), generator=g, device='cuda').half()
    wq, s = quant.symmetric_quantize(torch.randn((k, n), generator=g, device='cuda'), 'int8', 0)
    return x, wq, s.half(), torch.randn(n, generator=g, device='cuda').half()


@pytest.mark.parametrize('m,k,n', [(1, 512, 768), (16, 1024, 512), (70, 256, 320)])
def test_front_equals_the_python_path(m, k, n):
    announce('front', m, k, n)
    x, wq, s, b = _case(m, k, n)
    wide = torch.randn((m, k + 64), device='cuda').half()[:, :k]  # rows further apart than K
    nk = quant.to_decode_layout(wq)
    front = ffi.front()
    for a in (x, wide, x.reshape(1, m, k)):
        for w in (wq, nk):
            for bias in (None, b):
                got = quant.symmetric_quant_matmul(a, w, s, bias)
                assert torch.equal(got, run_w8a16(a, w, s, 0, bias)) and got.shape == a.shape[:-1] + (n,)
        assert front.w8a16(a, wq, s, None) is not None and (front.w8a16(a, nk, s, None) is not None) == (m <= 16)
    packed, gs = quant.symmetric_group_quantize_int4(torch.randn((k, n), device='cuda'), 128, 'float16')
    for bias in (None, b):
        assert torch.equal(quant.symmetric_quant_matmul_w4a16(wide, packed, gs, 128, bias), _run_w4a16(wide, packed, gs, 128, bias))
    a8, sa = F8.fp8_quantize_per_tensor(x)
    b8, sb = F8.fp8_quantize_per_tensor(torch.randn((n, k), device='cuda'))
    assert torch.equal(F8.matmul_f8_per_tensor(a8, b8, sa, sb), F8._run_f8(a8, b8, torch.bfloat16, sa, sb))
    for _ in range(2):
        assert torch.equal(F8.matmul_f8(a8, b8, output_dtype='float32'), F8._run_f8(a8, b8, torch.float32))


@pytest.mark.parametrize('shape,dim', [((96, 200), 0), ((33, 260), -1), ((3, 40, 24), [1]), ((3, 40, 24), 0)])
def test_quantizers_equal_the_python_path(shape, dim):
    announce('front quantizers', shape, dim)
    w = torch.randn(shape, device='cuda')
    for dtype in (torch.float32, torch.bfloat16):
        for codes in ('int8', 'int16'):
            q, s = quant.symmetric_quantize(w.to(dtype), codes, dim)
            op = symmetric.SymmetricQuantizationOp(w.to(dtype), getattr(torch, codes), dims=dim)
            assert torch.equal(q, op.outputs[0]) and torch.equal(s, op.outputs[1])
            assert torch.equal(quant.symmetric_dequantize(q, s, dim), symmetric.SymmetricDeQuantizationOp(q, s, dim).outputs[0])


def test_int4_and_block_scaled_equal_the_python_path():
    announce('front int4 and block scaled')
    w = torch.randn((512, 264), device='cuda')
    p, s = quant.symmetric_group_quantize_int4(w, 128, 'bfloat16')
    op = group_int4.SymmetricGroupQuantizationInt4Op(w, 128, torch.bfloat16)
    assert torch.equal(p, op.outputs[0]) and torch.equal(s, op.outputs[1])
    x, nk = torch.randn((3, 512), device='cuda').bfloat16(), quant.to_decode_layout_int4(p)
    out = quant.symmetric_quant_matmul_w4a16_decode(x, nk, s)
    # the same values through a view that the front leaves to Python (no 16-byte aligned rows)
    assert torch.equal(out, quant.symmetric_quant_matmul_w4a16_decode(torch.nn.functional.pad(x, (1, 0))[:, 1:], nk, s))
    a, b = torch.randn((40, 256), device='cuda').to(F8.f8e4m3), torch.randn((384, 256), device='cuda').to(F8.f8e4m3)
    sa, sb = torch.rand((2, 40), device='cuda'), torch.rand((3, 2), device='cuda')
    want = F8.MatmulF8ScaledOperator(a, b, sa, sb, torch.float32, torch.bfloat16).outputs[0]
    assert torch.equal(F8.matmul_f8_scaled(a, b, sa, sb, output_dtype='bfloat16'), want)


def test_what_the_front_leaves_to_python():
    announce('front: left to Python')
    x, wq, s, b = _case(4, 256, 512)
    front = ffi.front()
    sparse_rows = torch.randn((4, 512), device='cuda').half()[:, ::2]
    for args in ((x.float(), wq, s, None), (x, wq.t(), s, None), (x, wq, s.float(), None), (x, wq, s, b[:8]), (x[:, :128], wq, s, None),
                 (sparse_rows, wq, s, None), (x.cpu(), wq, s, None), (x, wq, s.cpu(), None), (x[0], wq, s, None), (x[:0], wq, s, None)):
        assert front.w8a16(*args) is None
    assert torch.equal(quant.symmetric_quant_matmul(sparse_rows, wq, s), quant.symmetric_quant_matmul(sparse_rows.contiguous(), wq, s))
    assert quant.symmetric_quant_matmul(x[:0], wq, s).shape == (0, 512)
    with pytest.raises(ValueError):
        quant.symmetric_quant_matmul(x.float(), wq, s)
    with pytest.raises(BackendException):
        quant.symmetric_quant_matmul(x, wq, s.cpu())
    for axis in (2, -3, 2 ** 70):
        assert front.quantize(x, torch.int8, axis) is None
        with pytest.raises((ValueError, IndexError)):
            quant.symmetric_quantize(x, 'int8', axis)
    ffi.load_library().hidet_set_last_error(b'planted')  # an error the library reports surfaces as the exception
    with pytest.raises(BackendException, match='planted'):
        quant.symmetric_quant_matmul(x, wq, s)


def test_each_stream_has_its_workspace():
    announce('front: streams')
    x, wq, s, _ = _case(2, 4096, 8192)
    want = quant.symmetric_quant_matmul(x, wq, s)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        got = quant.symmetric_quant_matmul(x, wq, s)
        assert (x.device.index, stream.cuda_stream) in ffi._WORKSPACES
    stream.synchronize()
    assert torch.equal(got, want)


def test_a_missing_scale_is_an_error():
    announce('front: missing scales')
    a, sa = F8.fp8_quantize_per_tensor(torch.randn((3, 64), device='cuda'))
    b, sb = F8.fp8_quantize_per_tensor(torch.randn((32, 64), device='cuda'))
    for scales in ((None, sb), (sa, None), (None, None)):
        with pytest.raises(AttributeError):
            F8.matmul_f8_per_tensor(a, b, *scales)
    for scales in ((None, sb), (sa, None)):
        assert ffi.front().matmul_f8(a, b, *scales, torch.float32) is None
    assert torch.equal(ffi.front().matmul_f8(a, b, None, None, torch.float32), F8.matmul_f8(a, b, output_dtype='float32'))


def test_a_group_size_no_integer_type_holds():
    announce('front: group sizes')
    w = torch.randn((256, 64), device='cuda')
    p, s = quant.symmetric_group_quantize_int4(w, 128, 'float16')
    x, nk, front = torch.randn((2, 256), device='cuda').half(), quant.to_decode_layout_int4(p), ffi.front()
    for group in (2 ** 70, -2 ** 70, 2 ** 40, -1, 0):
        assert front.quantize_int4(w, group, torch.float16) is None and front.w4a16(x, p, s, group, None) is None
        assert front.w4a16_decode(x, nk, s, group) is None
    for call in (lambda: quant.symmetric_group_quantize_int4(w, 2 ** 70), lambda: quant.symmetric_quant_matmul_w4a16(x, p, s, 2 ** 70),
                 lambda: quant.symmetric_quant_matmul_w4a16_decode(x, nk, s, 2 ** 70)):
        with pytest.raises((ValueError, AssertionError)):
            call()


def test_an_error_names_the_entry_point_and_the_arguments():
    announce('front: errors')
    x, wq, s, b = _case(2, 256, 512)
    nk, lib = quant.to_decode_layout(wq), ffi.load_library()
    for w, bias, name in ((wq, None, 'i8'), (wq, b, 'i8_bias'), (nk, None, 'i8_nk'), (nk, b, 'i8_nk_bias')):
        lib.hidet_set_last_error(b'planted')
        with pytest.raises(BackendException) as e:
            quant.symmetric_quant_matmul(x, w, s, bias)
        text = str(e.value)
        assert 'Calling hidet_symmetric_quant_matmul_f16_' + name + ' with' in text and 'planted' in text
        assert 'shape=(2, 256), dtype=torch.float16' in text and text.endswith(ffi.LIB_PATH)
    with pytest.raises(BackendException, match=r'shape=\(32, 64\)(.|\n)*8-byte aligned'):  # the library's own check
        quant.symmetric_group_quantize_int4(torch.randn(32 * 64 + 1, device='cuda')[1:].view(32, 64), 32)
