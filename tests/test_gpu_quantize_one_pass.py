"""symmetric_quantize in one pass over the weight (strips of columns, workgroups that meet): bit-exact against the oracle at the edges of
the rows that the kernels hold, of their column blocks and of the sizes between which the operator chooses."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, host
from test_gpu_quantize_edges import _near_ties

pytestmark = pytest.mark.gpu


def _matrix(shape, dim, codes, dtype):
    w = _near_ties(np.random.default_rng(shape[-1]), shape, dim, 127 if codes == 'int8' else 32767)
    w.reshape(-1, shape[-1])[:, -1] = 0  # a column of zeros, in the quad that may be moved back into the row
    w.reshape(-1, shape[-1])[-1, 0] = 3.0  # a maximum in the last row
    if dtype == 'bfloat16':
        w = O.to_bf16(w)
    elif dtype == 'float16':
        w = w.astype(np.float16)
    return w, O.symmetric_quantize(w, codes, dim, dtype=dtype, target='cpu' if dtype == 'float32' else 'gpu')


def _check(got, want):
    assert np.array_equal(host(got[0]), want[0])
    assert np.array_equal(got[1].float().cpu().numpy(), np.asarray(want[1], dtype=np.float32))


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('shape,dim,codes', [
    # strips of 8, 16 and 32 columns: rows held, one more, the last that take this kernel; columns that end in part of a quad
    ((2, 97), 0, 'int8'), ((1024, 98), 0, 'int16'), ((1025, 2048), 0, 'int8'), ((1536, 99), 0, 'int8'), ((1536, 2052), 0, 'int8'), ((2048, 2051), 0, 'int16'),
    ((513, 4098), 0, 'int8'), ((1024, 4101), 0, 'int8'), ((640, 8194), 0, 'int16'), ((3, 300, 201), 1, 'int8'),
    # workgroups that meet: a last range of one row, 8, 16 and 20 quads held (and 8 in LDS), rows beyond those, slices
    ((1537, 1030), 0, 'int8'), ((1921, 2050), 0, 'int16'), ((4096, 1539), 0, 'int8'), ((4095, 4098), 0, 'int8'), ((3000, 6401), 0, 'int8'), ((15000, 2052), 0, 'int16'),
    ((2, 2100, 1301), 1, 'int8')])
def test_bit_exact(shape, dim, codes, dtype):
    announce('quantize in one pass', shape, dim, codes, dtype)
    w, want = _matrix(shape, dim, codes, dtype)
    _check(quant.symmetric_quantize(dev(w).to(getattr(torch, dtype)), codes, dim), want)


@pytest.mark.parametrize('shape', [(2048, 2050), (4096, 2100)])
def test_workgroups_that_do_not_wait(shape):
    # a limit of zero polls: whoever is not the last of its column block reads the whole block itself
    announce('quantize in one pass: poll limit 0', shape)
    w, want = _matrix(shape, 0, 'int8', 'float32')
    x = dev(w)
    lib = ffi.load_library()
    lib.hidet_qmm_set_exchange_spin_limit(0)
    try:
        for _ in range(3):
            _check(quant.symmetric_quantize(x, 'int8', 0), want)
    finally:
        lib.hidet_qmm_set_exchange_spin_limit(-1)
    assert not ffi.workspace(x.device)[:65536].any()  # the counters are back at zero
    _check(quant.symmetric_quantize(x, 'int8', 0), want)


def test_replayed_graph():
    announce('quantize in one pass: graph')
    w, want = _matrix((2048, 2050), 0, 'int8', 'float32')
    x = dev(w)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        quant.symmetric_quantize(x, 'int8', 0)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = quant.symmetric_quantize(x, 'int8', 0)
    for _ in range(4):
        got[0].zero_(), got[1].zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(got, want)
        quant.symmetric_quantize(x, 'int8', 0)
