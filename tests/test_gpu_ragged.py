"""Sizes off the matrix kernels' tiles: N a multiple of 4 (int4: 8) only, where the last lane with columns shares some of them
with its neighbour, and K or N that the matrix kernels do not take at all, where they run on padded copies. Small integers and
powers of two: every sum is exact, the result must equal integer arithmetic with the definition's roundings, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, fastest_ms, host

pytestmark = pytest.mark.gpu


def _int8_case(m, k, n, biased):
    rng = np.random.default_rng(1000 * m + k + n)
    a = rng.integers(-3, 4, (m, k)).astype(np.float32)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    s = (2.0 ** rng.integers(-6, 1, n)).astype(np.float32)
    with np.errstate(over='ignore'):
        want = ((a.astype(np.float64) @ w.astype(np.float64)) * s).astype(np.float32).astype(np.float16)
        b = (rng.integers(-64, 65, n) / 8.0).astype(np.float16) if biased else None
        if biased:
            want = (want.astype(np.float32) + b.astype(np.float32)).astype(np.float16)
    return dev(a.astype(np.float16)), dev(w), dev(s.astype(np.float16)), None if b is None else dev(b), want


@pytest.mark.parametrize('m,k,n,biased', [
    # N a multiple of 4: one short lane in the first tile, a tile of 4 columns behind a whole one, both exchange layouts, K tails
    (1, 96, 20, False), (3, 4096, 260, True), (16, 4100, 516, False), (1, 4096, 8196, False), (2, 1002, 8204, True), (24, 2050, 276, False),
    # padded copies: N of no multiple of 4 with one pass of 16 rows and with the GEMM, K of no multiple of 64, several row tiles
    (1, 4100, 258, False), (16, 1022, 1030, True), (17, 4094, 518, False), (33, 4100, 260, True), (129, 1000, 770, False), (300, 2050, 4098, True)])
def test_int8_exact(m, k, n, biased):
    announce('ragged int8', m, k, n, biased)
    a, w, s, b, want = _int8_case(m, k, n, biased)
    for _ in range(2):  # the exchange's mailbox is clean again after the first call
        assert np.array_equal(host(quant.symmetric_quant_matmul(a, w, s, b)), want)


# N = 4 i + 2 on the narrow tiles as it lies: one column pair to spare, one short of a tile and one more, two tiles and a pair; one to three
# row blocks per wave group, K of less than a stage, of several pieces, ending inside a stage. Rows of the activations are followed by NaN, which
# the last stage's reads bring along.
@pytest.mark.parametrize('m,k,n,biased', [(1, 64, 2, False), (3, 66, 6, True), (17, 26, 4094, False), (1, 16390, 122, True), (2, 4096, 126, False), (16, 4098, 250, True), (33, 1030, 374, False),
                                          (64, 2048, 1022, True), (65, 994, 2050, False), (128, 1000, 126, True), (131, 3000, 498, False), (1000, 130, 4098, True)])
def test_int8_rows_off_the_dwords(m, k, n, biased):
    announce('ragged int8 off the dwords', m, k, n, biased)
    a, w, s, b, want = _int8_case(m, k, n, biased)
    wide = torch.full((m, k + 6), float('nan'), dtype=torch.float16, device='cuda')
    wide[:, :k] = a
    ws = ffi.workspace(a.device)
    for _ in range(2):
        c = torch.full((m + 1, n), 7.0, dtype=torch.float16, device='cuda')
        args = (wide, w, s, b, c) if biased else (wide, w, s, c)
        ffi.call('hidet_symmetric_quant_matmul_f16_i8' + ('_bias' if biased else ''), *args, m, k, n, k + 6, 0, ws, ws.numel(), ffi.current_stream(a.device))
        assert np.array_equal(host(c[:m]), want) and bool((c[m] == 7.0).all())


@pytest.mark.parametrize('scratch', [1 << 20, 3 << 20])
def test_int8_in_panels_of_a_small_workspace(scratch):
    announce('ragged int8 panels', scratch)
    m, k, n = 270, 1000, 1031
    a, w, s, _, want = _int8_case(m, k, n, False)
    c = torch.empty((m, n), dtype=torch.float16, device='cuda')
    ws = torch.zeros(int(ffi.load_library().hidet_qmm_workspace_bytes_for_scratch(scratch)), dtype=torch.uint8, device='cuda')
    ffi.call('hidet_symmetric_quant_matmul_f16_i8', a, w, s, c, m, k, n, k, 0, ws, ws.numel(), ffi.current_stream(a.device))
    assert np.array_equal(host(c), want)


# up to 16 rows of a weight whose padded copy does not fit the workspace whole: panels, as for more rows
@pytest.mark.parametrize('m,k,n,biased', [(1, 1000, 1031, False), (16, 1022, 4099, True), (3, 256, 9002, True)])
def test_int8_decode_in_panels_of_a_small_workspace(m, k, n, biased):
    announce('ragged int8 decode panels', m, k, n, biased)
    a, w, s, b, want = _int8_case(m, k, n, biased)
    ws = torch.zeros(int(ffi.load_library().hidet_qmm_workspace_bytes_for_scratch(1 << 20)), dtype=torch.uint8, device='cuda')
    for _ in range(2):
        c = torch.empty((m, n), dtype=torch.float16, device='cuda')
        args = (a, w, s, b, c) if biased else (a, w, s, c)
        ffi.call('hidet_symmetric_quant_matmul_f16_i8' + ('_bias' if biased else ''), *args, m, k, n, k, 0, ws, ws.numel(), ffi.current_stream(a.device))
        assert np.array_equal(host(c), want)


@pytest.mark.parametrize('m', [1, 16])
def test_int8_decode_of_a_large_ragged_weight_costs_no_more_than_more_rows(m):
    """8192 x 8190 does not fit the standing workspace: in panels it takes what 17 rows take, element by element fifty times that."""
    announce('ragged int8 decode, large', m)
    k, n = 8192, 8190
    w = torch.randint(-7, 8, (k, n), device='cuda', dtype=torch.int8)
    x = torch.randint(-3, 4, (17, k), device='cuda').half()
    s = torch.ones(n, device='cuda', dtype=torch.float16)

    want = (x.float() @ w.float()).half()
    assert torch.equal(quant.symmetric_quant_matmul(x[:m], w, s), want[:m])
    assert fastest_ms(lambda: quant.symmetric_quant_matmul(x[:m], w, s)) < 8 * fastest_ms(lambda: quant.symmetric_quant_matmul(x, w, s))


def test_int8_off_the_dwords_without_room_for_a_copy():
    """N = 4 i + 2 where the prefill tiles would be estimated faster on a padded copy that the workspace has no room for: on the narrow
    tiles as it lies (element by element a hundred times slower)."""
    announce('ragged int8 off the dwords, no room')
    m, k, n = 1000, 4096, 4098
    w = torch.randint(-7, 8, (k, n), device='cuda', dtype=torch.int8)
    x = torch.randint(-3, 4, (m, k), device='cuda').half()
    s = torch.ones(n, device='cuda', dtype=torch.float16)
    c = torch.empty((m, n), dtype=torch.float16, device='cuda')
    small = torch.zeros(int(ffi.load_library().hidet_qmm_workspace_bytes_for_scratch(1 << 16)), dtype=torch.uint8, device='cuda')

    def call():
        ffi.call('hidet_symmetric_quant_matmul_f16_i8', x, w, s, c, m, k, n, k, 0, small, small.numel(), ffi.current_stream(x.device))

    call()
    assert torch.equal(c, (x.float() @ w.float()).half())
    assert fastest_ms(call) < 8 * fastest_ms(lambda: quant.symmetric_quant_matmul(x, w, s))


@pytest.mark.parametrize('m,k,n,group', [(1, 256, 24, 128), (16, 4096, 264, 128), (3, 1024, 1032, 32), (20, 512, 520, 64)])
def test_int4_exact(m, k, n, group):
    announce('ragged int4', m, k, n, group)
    rng = np.random.default_rng(m + k + n)
    a = rng.integers(-3, 4, (m, k)).astype(np.float32)
    q = rng.integers(-7, 8, (k, n)).astype(np.int8)
    s = rng.integers(1, 4, (k // group, n)).astype(np.float32)
    want = O.to_bf16((a.astype(np.float64) @ (q.astype(np.float64) * np.repeat(s, group, axis=0))).astype(np.float32))
    got = quant.symmetric_quant_matmul_w4a16(dev(a, torch.bfloat16), dev(O.pack_int4(q)), dev(s, torch.bfloat16), group)
    assert np.array_equal(host(got), want)


# K odd, rows of an even stride (what a C caller may pass): the last element of the last row counts, the one behind it does not
@pytest.mark.parametrize('m,k,n', [(17, 129, 256), (31, 4097, 260), (33, 1001, 512), (64, 63, 1024), (130, 2047, 388)])
def test_int8_odd_k(m, k, n):
    announce('ragged int8 odd k', m, k, n)
    a, w, s, _, _ = _int8_case(m, k, n, False)
    a[-1, -1], w[-1] = 3, 100
    wide = torch.full((m, k + 1), float('nan'), dtype=torch.float16, device='cuda')
    wide[:, :k] = a
    want = ((a.double() @ w.double()) * s.double()).float().half()
    c = torch.empty((m, n), dtype=torch.float16, device='cuda')
    ws = ffi.workspace(a.device)
    ffi.call('hidet_symmetric_quant_matmul_f16_i8', wide, w, s, c, m, k, n, k + 1, 0, ws, ws.numel(), ffi.current_stream(a.device))
    assert torch.equal(c, want)


def test_int8_rows_beyond_31_bit_offsets():
    """So wide that 160 rows of the weight take more than 2 GiB, N no multiple of 4: neither the bandwidth-bound kernel nor its
    padded copies can address it."""
    m, k, n = 1, 2, 13_500_002
    announce('ragged int8 wide', m, k, n)
    g = torch.Generator(device='cuda').manual_seed(3)
    a = torch.tensor([[3.0, -2.0]], device='cuda').half()
    w = torch.randint(-127, 128, (k, n), generator=g, device='cuda', dtype=torch.int8)
    s = torch.full((n,), 0.5, device='cuda', dtype=torch.float16)
    want = ((3.0 * w[0].float() - 2.0 * w[1].float()) * 0.5).half()[None]
    c = torch.empty((m, n), dtype=torch.float16, device='cuda')
    for scratch in (64 << 20, 160 << 20):  # without and with room for a copy of the weight
        ws = torch.zeros(int(ffi.load_library().hidet_qmm_workspace_bytes_for_scratch(scratch)), dtype=torch.uint8, device='cuda')
        ffi.call('hidet_symmetric_quant_matmul_f16_i8', a, w, s, c, m, k, n, k, 0, ws, ws.numel(), ffi.current_stream(a.device))
        assert torch.equal(c, want)
