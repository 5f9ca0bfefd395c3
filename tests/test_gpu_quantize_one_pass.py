"""symmetric_quantize in one pass over the weight (strips of columns, workgroups that meet): bit-exact against the oracle at the edges of
the rows that the kernels hold, of their column blocks and of the sizes between which the operator chooses."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, host, last_launch, variant
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


def _launched(dtype, codes, kernel):
    """`kernel`: ('strip', column quads) or ('meet', quads held of float32 or twice as many 16-bit ones, quads in LDS of float32)."""
    types, wide = [ffi.DTYPE_CODE[getattr(torch, dtype)], ffi.DTYPE_CODE[getattr(torch, codes)]], 1 if dtype == 'float32' else 2
    name = last_launch()[0]
    if kernel[0] == 'strip':
        assert variant('quantize_strip_kernel', *types, kernel[1])[:-1] in name, name
    else:
        assert variant('quantize_meet_kernel', *types, wide * kernel[1], kernel[2] if wide == 1 else 0) in name, name


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('shape,dim,codes,kernel,kernel_16', [
    # strips of 8, 16 and 32 columns: rows held, one more, the last that take this kernel; columns that end in part of a quad
    ((2, 97), 0, 'int8', ('strip', 2), None), ((1024, 98), 0, 'int16', ('strip', 2), None), ((1025, 2048), 0, 'int8', ('strip', 2), None),
    ((1536, 99), 0, 'int8', ('strip', 2), None), ((1536, 2052), 0, 'int8', ('strip', 4), None), ((2048, 2051), 0, 'int16', ('strip', 4), ('meet', 8, 0)),
    ((513, 4098), 0, 'int8', ('strip', 8), None), ((1024, 4101), 0, 'int8', ('strip', 8), None), ((640, 8194), 0, 'int16', ('strip', 8), None),
    ((3, 300, 201), 1, 'int8', ('strip', 2), None),
    # workgroups that meet: a last range of one row, 8, 16 and 20 quads held (and 8 in LDS), rows beyond those, slices
    ((1537, 1030), 0, 'int8', ('meet', 8, 0), None), ((1921, 2050), 0, 'int16', ('strip', 4), ('meet', 8, 0)), ((2049, 2050), 0, 'int16', ('meet', 16, 0), ('meet', 8, 0)),
    ((4096, 1539), 0, 'int8', ('meet', 16, 0), ('meet', 8, 0)), ((4095, 4098), 0, 'int8', ('meet', 20, 8), ('meet', 16, 0)),
    ((3000, 6401), 0, 'int8', ('meet', 20, 8), ('meet', 16, 0)), ((15000, 2052), 0, 'int16', ('meet', 20, 8), ('meet', 20, 0)),
    ((2, 2100, 1301), 1, 'int8', ('meet', 16, 0), ('meet', 8, 0))])
def test_bit_exact(shape, dim, codes, kernel, kernel_16, dtype):
    announce('quantize in one pass', shape, dim, codes, dtype)
    w, want = _matrix(shape, dim, codes, dtype)
    got = quant.symmetric_quantize(dev(w).to(getattr(torch, dtype)), codes, dim)
    _launched(dtype, codes, kernel if dtype == 'float32' or kernel_16 is None else kernel_16)
    _check(got, want)


# quads held in registers, in LDS too, rows beyond those, 16-bit types, several slices
MEETINGS = [((2049, 2050), 0, 'int8', 'float32'), ((1537, 1030), 0, 'int16', 'float32'), ((3000, 6401), 0, 'int8', 'float32'), ((15000, 2052), 0, 'int8', 'float32'),
            ((2, 2100, 1301), 1, 'int8', 'float32'), ((4096, 2100), 0, 'int8', 'bfloat16'), ((15000, 2052), 0, 'int16', 'float16')]


@pytest.mark.parametrize('shape,dim,codes,dtype', MEETINGS)
def test_workgroups_that_do_not_wait(shape, dim, codes, dtype):
    # a limit of zero polls: whoever is not the last of its column block reads the whole block itself
    announce('quantize in one pass: poll limit 0', shape, codes, dtype)
    w, want = _matrix(shape, dim, codes, dtype)
    x = dev(w).to(getattr(torch, dtype))
    lib = ffi.load_library()
    lib.hidet_qmm_set_exchange_spin_limit(0)
    try:
        for _ in range(3):
            _check(quant.symmetric_quantize(x, codes, dim), want)
            assert 'quantize_meet_kernel' in last_launch()[0]
    finally:
        lib.hidet_qmm_set_exchange_spin_limit(-1)
    assert not ffi.workspace(x.device)[:65536].any()  # the counters are back at zero
    _check(quant.symmetric_quantize(x, codes, dim), want)


def test_scratch_for_the_maxima_alone():
    # no room for what the workgroups leave each other: the two launches of before
    announce('quantize in one pass: little scratch')
    w, want = _matrix((2049, 2050), 0, 'int8', 'float32')
    x, q, s = dev(w), torch.empty((2049, 2050), dtype=torch.int8, device='cuda'), torch.empty(2050, device='cuda')
    ws = torch.zeros(ffi.load_library().hidet_qmm_workspace_bytes_for_scratch(4 * 2050), dtype=torch.uint8, device='cuda')
    ffi.call('hidet_symmetric_quantize', x, q, s, 1, 2049, 2050, ffi.F32, ffi.I8, ws, ws.numel(), ffi.current_stream(x.device))
    assert 'quantize_meet' not in last_launch()[0] and 'quantize_strip' not in last_launch()[0]
    _check((q, s), want)


def test_meetings_on_two_streams():
    announce('quantize in one pass: two streams')
    cases = [_matrix((4096, 2100), 0, 'int8', 'float32'), _matrix((3000, 6401), 0, 'int8', 'float32')]
    xs, streams, got = [dev(w) for w, _ in cases], [torch.cuda.Stream(), torch.cuda.Stream()], [[], []]
    torch.cuda.synchronize()
    for _ in range(20):
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                got[i].append(quant.symmetric_quantize(xs[i], 'int8', 0))
                assert 'quantize_meet_kernel' in last_launch()[0]
    torch.cuda.synchronize()
    for i, (_, want) in enumerate(cases):
        for g in got[i]:
            _check(g, want)
    for stream in streams:
        with torch.cuda.stream(stream):
            assert not ffi.workspace(xs[0].device)[:65536].any()


@pytest.mark.parametrize('shape,dim,codes,dtype', [((2048, 2050), 0, 'int8', 'float32')] + MEETINGS)
def test_replayed_graph(shape, dim, codes, dtype):
    announce('quantize in one pass: graph', shape, codes, dtype)
    w, want = _matrix(shape, dim, codes, dtype)
    x = dev(w).to(getattr(torch, dtype))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        quant.symmetric_quantize(x, codes, dim)
        assert ('quantize_meet_kernel' in last_launch()[0]) == (shape != (2048, 2050))
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = quant.symmetric_quantize(x, codes, dim)
        workspace = ffi.workspace(x.device)
    for _ in range(4):
        got[0].zero_(), got[1].zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(got, want)
        quant.symmetric_quantize(x, codes, dim)
    torch.cuda.synchronize()
    assert not workspace[:65536].any()
