"""The narrow-tile GEMMs that serve 17 to about 1000 rows, at the edges of their tiles, K stages and K splits.

Operands are small integers and the column factors powers of two, so that every product and sum is exact in float32 and the
only rounding is that of the result: the expected values are computed in float64 and rounded the same way."""
import pytest
import torch

from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from hidet_amd.graph.ops.matmul import matmul_f8 as f8
from gpu_util import announce, fastest_ms, last_launch

pytestmark = pytest.mark.gpu


def _ints(g, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=g, device='cuda')


# rows around the 32 / 64 / 128 of the tiles; K off the 32 of a stage (and odd multiples of 2), from less than one stage to
# eight pieces; N off the 128 of a tile, down to one chunk
@pytest.mark.parametrize('m,k,n', [(17, 256, 4), (31, 4098, 132), (32, 64, 128), (33, 96, 260), (48, 64, 64), (64, 11008, 516), (65, 34, 516),
                                   (70, 66, 20), (127, 1000, 1028), (129, 4096, 384), (203, 4100, 4098), (512, 4096, 1024),
                                   (300, 96, 200), (700, 2048, 4096)])
def test_w8a16_rows_of_a_batch(m, k, n):
    g = torch.Generator(device='cuda')
    g.manual_seed(m * 31 + k + n)
    x, w = _ints(g, (m, k), -3, 3).half(), _ints(g, (k, n), -7, 7).to(torch.int8)
    scale = (2.0 ** _ints(g, (n,), -4, 0).float()).half()
    bias = _ints(g, (n,), -4, 4).half()
    want = ((x.double() @ w.double()) * scale.double()).half()
    layouts = [w]
    if m <= 64 and k % 64 == 0 and n % 4 == 0:
        layouts.append(quant.to_decode_layout(w))
    for weight in layouts:
        for _ in range(2):  # the exchange's counters are back at zero for the second call
            assert torch.equal(quant.symmetric_quant_matmul(x, weight, scale), want)
        assert torch.equal(quant.symmetric_quant_matmul(x, weight, scale, bias), (want.float() + bias.float()).half())


def test_w8a16_values_past_k_do_not_reach_the_result():
    """A K stage that ends inside the matrix reads the next row's activations too: NaN and infinities there stay out."""
    g = torch.Generator(device='cuda')
    g.manual_seed(5)
    m, k, n = 40, 70, 256
    wide = torch.full((m, 96), float('nan'), device='cuda', dtype=torch.float16)
    wide[:, ::2] = float('inf')
    wide[:, :k] = _ints(g, (m, k), -3, 3).half()
    x, w = wide[:, :k], _ints(g, (k, n), -7, 7).to(torch.int8)
    scale = torch.ones(n, device='cuda', dtype=torch.float16)
    assert torch.equal(quant.symmetric_quant_matmul(x, w, scale), (x.double() @ w.double()).half())


# rows around the 32 / 64 of the tiles; K of less than one 128-deep stage, off the stages (multiples of 16), of many pieces; N
# off the 128 of a tile
@pytest.mark.parametrize('m,k,n', [(17, 128, 4), (31, 144, 60), (33, 272, 132), (64, 4096, 4096), (65, 1040, 516), (100, 16, 4), (200, 2048, 68),
                                   (256, 7168, 640), (1000, 512, 256)])
def test_fp8_rows_of_a_batch(m, k, n):
    g = torch.Generator(device='cuda')
    g.manual_seed(m + k + n)
    a, b = _ints(g, (m, k), -3, 3).float().to(torch.float8_e4m3fn), _ints(g, (n, k), -3, 3).float().to(torch.float8_e4m3fn)
    half, quarter = torch.tensor(0.5, device='cuda'), torch.tensor(0.25, device='cuda')
    exact = (a.double() @ b.double().t()) * 0.125
    for dtype in (torch.float32, torch.float16, torch.bfloat16, torch.float32):
        assert torch.equal(f8.matmul_f8_per_tensor(a, b, half, quarter, output_dtype=dtype), exact.to(dtype))


@pytest.mark.parametrize('m,k,n', [(17, 128, 128), (64, 7168, 512), (65, 1024, 256), (130, 2048, 1536), (513, 512, 384)])
def test_fp8_block_scaled_rows_of_a_batch(m, k, n):
    g = torch.Generator(device='cuda')
    g.manual_seed(m + k + n)
    a, b = _ints(g, (m, k), -3, 3).float().to(torch.float8_e4m3fn), _ints(g, (n, k), -3, 3).float().to(torch.float8_e4m3fn)
    scale_a, scale_b = 2.0 ** _ints(g, (k // 128, m), -3, 0).float(), 2.0 ** _ints(g, (n // 128, k // 128), -3, 0).float()
    af = (a.double().view(m, k // 128, 128) * scale_a.t().double()[:, :, None]).view(m, k)
    bf = (b.double().view(n // 128, 128, k // 128, 128) * scale_b.double()[:, None, :, None]).view(n, k)
    want = (af @ bf.t()).float()
    for _ in range(2):
        assert torch.equal(f8.matmul_f8_scaled(a, b, scale_a, scale_b, output_dtype='float32'), want)


def _int4(g, k, n, group, dtype):
    """Packed codes of small integers with scales that are powers of two, and the weights they stand for."""
    q = _ints(g, (k, n), -8, 7)
    packed = ((q[:, 0::2] & 0xF) | ((q[:, 1::2] & 0xF) << 4)).to(torch.uint8)
    scales = 2.0 ** _ints(g, (k // group, n), -3, 0).double()
    return packed, scales.to(dtype), q.double() * scales.repeat_interleave(group, 0)


# rows around the 32 / 64 of the tiles, K of one 32-deep stage and of many pieces, N off the 128 of a tile, every kind of group
@pytest.mark.parametrize('m,k,n,group', [(17, 32, 8, 32), (31, 128, 136, 128), (33, 192, 1032, 64), (64, 11008, 264, 128), (65, 96, 72, 96), (70, 4096, 4096, 128),
                                         (200, 2048, 520, 64), (300, 512, 128, 256)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_w4a16_rows_of_a_batch(m, k, n, group, dtype):
    g = torch.Generator(device='cuda')
    g.manual_seed(m + k + n)
    x = _ints(g, (m, k), -2, 2).to(dtype)
    packed, scales, w = _int4(g, k, n, group, dtype)
    want = (x.double() @ w).to(dtype)
    for _ in range(2):
        assert torch.equal(quant.symmetric_quant_matmul_w4a16(x, packed, scales, group), want)


# 64-deep stages (groups of 64 and its multiples): one, two and an odd number of stages, fewer and more of them than the ring holds, a group a stage
# and several, pieces of K that begin inside a group; one chunk of columns. Groups of an odd number of 32 beside them.
@pytest.mark.parametrize('m,k,n,group', [(17, 64, 8, 64), (33, 128, 136, 64), (64, 128, 8, 128), (40, 960, 264, 192), (65, 8256, 120, 64), (100, 11008, 1032, 256),
                                         (128, 1152, 2056, 128), (40, 1248, 264, 96), (65, 160, 8, 160),
                                         # 32 rows a tile, groups of 64 and more: 32-deep stages by their estimate (one to eight pieces of K), 64-deep ones
                                         (17, 64, 1032, 64), (26, 1408, 2240, 128), (20, 1984, 136, 64), (31, 6528, 1448, 192), (96, 1024, 4096, 128), (128, 2560, 4096, 128)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_w4a16_depths_of_a_stage(m, k, n, group, dtype):
    announce('int4 stages', m, k, n, group, dtype)
    test_w4a16_rows_of_a_batch(m, k, n, group, dtype)


# the tall tiles of 96 columns: N = 96 i, + 32 and + 64 (a lane's three columns lie across the end), part-filled and short row tiles, one stage, fewer
# and more of them than the rings hold
@pytest.mark.parametrize('m,k,n,group', [(512, 64, 11040, 64), (400, 192, 11072, 64), (385, 512, 11008, 128), (490, 1024, 12288, 128), (449, 256, 10016, 256),
                                         (250, 128, 24544, 128), (200, 320, 20000, 64)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_w4a16_tiles_of_96_columns(m, k, n, group, dtype):
    announce('int4 tiles of 96 columns', m, k, n, group, dtype)
    test_w4a16_rows_of_a_batch(m, k, n, group, dtype)


def test_w4a16_infinite_and_large_activations():
    g = torch.Generator(device='cuda')
    g.manual_seed(8)
    m, k, n = 40, 256, 128
    x = _ints(g, (m, k), -2, 2).to(torch.bfloat16)
    x[3, 17] = float('inf')
    x[4] = 0
    x[4, 0] = 2.0 ** 124
    packed, scales, w = _int4(g, k, n, 128, torch.bfloat16)
    want = (x.double() @ w).to(torch.bfloat16)  # row 3: infinities, NaN where the code is zero
    assert torch.equal(quant.symmetric_quant_matmul_w4a16(x, packed, scales, 128).nan_to_num(nan=-1.0), want.nan_to_num(nan=-1.0))


# groups that are no whole stages of the tall tiles, from where their general kernel took over; edges of the tiles in M and N
@pytest.mark.parametrize('m,k,n,group', [(192, 1024, 1032, 32), (257, 96, 264, 96), (513, 192, 136, 96), (1000, 256, 520, 32), (1024, 64, 8, 32)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_w4a16_small_groups_of_many_rows(m, k, n, group, dtype):
    test_w4a16_rows_of_a_batch(m, k, n, group, dtype)


def test_w4a16_small_groups_cost_no_more_than_large_ones():
    """Groups of 32 run on the narrow tiles wherever those are the faster; the general kernel took four times as long."""
    announce('w4a16 groups of 32')
    m, k, n = 512, 4096, 11008
    packed = torch.randint(0, 256, (k, n // 2), device='cuda', dtype=torch.uint8)
    x = torch.randn((m, k), device='cuda').bfloat16()
    scales = {group: torch.ones((k // group, n), device='cuda', dtype=torch.bfloat16) for group in (32, 128)}
    small, large = (fastest_ms(lambda: quant.symmetric_quant_matmul_w4a16(x, packed, scales[group], group)) for group in (32, 128))
    assert small < 2 * large


# a weight so wide that the tall tiles fill the chip: short matrices leave their empty row blocks out (one, two, three of four
# pairs of blocks at work), rows at both edges of each form, a last tile of 8 columns
@pytest.mark.parametrize('m', [17, 32, 33, 64, 65, 96, 97])
@pytest.mark.parametrize('nk', [False, True])
def test_w8a16_few_rows_of_a_wide_weight(m, nk):
    announce('wide w8a16', m, nk)
    k, n = 320, 131080
    g = torch.Generator(device='cuda').manual_seed(m)
    a = torch.randint(-3, 4, (m, k), generator=g, device='cuda').half()
    w = torch.randint(-7, 8, (k, n), generator=g, device='cuda', dtype=torch.int8)
    s = 2.0 ** torch.randint(-3, 1, (n,), generator=g, device='cuda').half()
    b = torch.randint(-8, 9, (n,), generator=g, device='cuda').half()
    want = ((a.float() @ w.float()) * s.float()).half()  # small integers: every sum and product is exact
    c = torch.empty((m, n), dtype=torch.float16, device='cuda')
    ws = ffi.workspace(a.device)
    weight = w.t().contiguous() if nk else w
    for bias in (None, b):
        name = 'hidet_symmetric_quant_matmul_f16_i8' + ('_nk' if nk else '') + ('_bias' if bias is not None else '')
        operands = (a, weight, s) + ((bias,) if bias is not None else ()) + (c,)
        ffi.call(name, *operands, m, k, n, k, k if nk else 0, ws, ws.numel(), ffi.current_stream(a.device))
        assert torch.equal(c, want if bias is None else (want.float() + b.float()).half())


# the same forms on padded copies: rows of the result that start anywhere and end inside a lane's columns
@pytest.mark.parametrize('m', [17, 50, 96])
def test_w8a16_few_rows_of_a_wide_ragged_weight(m):
    announce('wide ragged w8a16', m)
    k, n = 322, 131078
    g = torch.Generator(device='cuda').manual_seed(m)
    a = torch.randint(-3, 4, (m, k), generator=g, device='cuda').half()
    w = torch.randint(-7, 8, (k, n), generator=g, device='cuda', dtype=torch.int8)
    s = 2.0 ** torch.randint(-3, 1, (n,), generator=g, device='cuda').half()
    b = torch.randint(-8, 9, (n,), generator=g, device='cuda').half()
    want = ((a.float() @ w.float()) * s.float()).half()
    assert torch.equal(quant.symmetric_quant_matmul(a, w, s), want)
    assert torch.equal(quant.symmetric_quant_matmul(a, w, s, b), (want.float() + b.float()).half())


# Three pieces of K on 64-row tiles, although they take two turns of the chip (4 us less than whole tiles)
@pytest.mark.parametrize('m,k,n', [(171, 9600, 6016), (433, 9472, 2560)])
def test_w4a16_pieces_in_two_turns_of_the_chip(m, k, n):
    announce('int4: pieces in two turns', m, k, n)
    g = torch.Generator(device='cuda')
    g.manual_seed(m)
    packed, scales, w = _int4(g, k, n, 128, torch.bfloat16)
    x = _ints(g, (m, k), -1, 1).bfloat16()
    got = quant.symmetric_quant_matmul_w4a16(x, packed, scales, 128)
    name, workgroups, _ = last_launch()
    tiles = -(-m // 64) * -(-n // 128)
    assert 'gemm_mid_kernel' in name and workgroups == 8 * -(-3 * tiles // 8), (name, workgroups)
    assert torch.equal(got, (x.double() @ w).to(torch.bfloat16))


# Many row tiles read each weight of a narrow matrix: the memory's rate is no reason to leave them for the prefill tiles, which take 30 to 50 % longer
@pytest.mark.parametrize('m,k,n', [(467, 9472, 2176), (660, 6336, 1536), (505, 7360, 3712), (84, 6592, 10752)])
def test_w8a16_many_rows_of_a_narrow_deep_weight(m, k, n):
    announce('int8: many rows of a narrow deep weight', m, k, n)
    g = torch.Generator(device='cuda')
    g.manual_seed(m)
    x, w = _ints(g, (m, k), -1, 1).half(), _ints(g, (k, n), -4, 4).to(torch.int8)
    scale = (2.0 ** _ints(g, (n,), -4, 0).float()).half()
    got = quant.symmetric_quant_matmul(x, w, scale)
    assert 'gemm_mid_kernel' in last_launch()[0], last_launch()
    assert torch.equal(got, ((x.double() @ w.double()) * scale.double()).half())
