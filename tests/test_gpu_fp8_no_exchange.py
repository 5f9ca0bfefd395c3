"""FP8 matmuls of 17 and more rows of small weights, which one workgroup per column strip computes over all of K: several row tiles, waves without a step of K, K that ends inside a step, rows and columns past the end, every output type; and shapes next to them that stay with
the narrow tiles. Integer-valued codes and scales whose sums stay below 2^24: exact in float32, so the results must be equal."""
import numpy as np
import pytest
import torch

from hidet_amd.graph.ops.matmul import matmul_f8 as F8
from gpu_util import announce, dev, host, last_launch, variant
from test_gpu_fp8_tiles import operands

pytestmark = pytest.mark.gpu

# (17..32, 33..48, 49..64 rows of one tile; 65, 129 and 257 rows of several)
ROWS = [17, 32, 33, 48, 49, 64, 65, 97, 129, 257]


@pytest.mark.parametrize('m', ROWS)
@pytest.mark.parametrize('k,n', [(128, 4), (16, 132), (1024, 260), (1152, 1000), (1136, 2176), (2032, 1028), (2048, 2048), (4096, 8192)])
def test_per_tensor(m, k, n):
    announce('fp8 without exchange', m, k, n)
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, False)
    exact = (ai.astype(np.float32) @ bi.T.astype(np.float32)) * 0.5
    half, one = torch.full((), 0.5, device='cuda'), torch.ones((), device='cuda')
    for dtype in (torch.float32, torch.float16, torch.bfloat16) if m in (17, 97) else (torch.float32,):
        got = F8.matmul_f8_per_tensor(a, b, half, one, output_dtype=dtype)
        assert torch.equal(got.cpu(), torch.from_numpy(exact).to(dtype))


@pytest.mark.parametrize('m', ROWS)
@pytest.mark.parametrize('k,n', [(128, 128), (1024, 256), (1152, 1024), (7168, 512), (2048, 4096)])
def test_block_scaled(m, k, n):
    announce('block-scaled without exchange', m, k, n)
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, False)
    sa = rng.integers(1, 5, (k // 128, m)).astype(np.float32)
    sb = rng.integers(1, 5, (n // 128, k // 128)).astype(np.float32)
    exact = (ai * np.repeat(sa.T, 128, axis=1)).astype(np.float64) @ (bi * np.repeat(np.repeat(sb, 128, axis=0), 128, axis=1)).T.astype(np.float64)
    assert np.abs(exact).max() < 2 ** 24
    for dtype in ('float32', 'float16', 'bfloat16') if m in (17, 97) else ('float32',):
        got = F8.matmul_f8_scaled(a, b, scale_a=dev(sa), scale_b=dev(sb), output_dtype=dtype)
        assert torch.equal(got.cpu(), torch.from_numpy(exact.astype(np.float32)).to(getattr(torch, dtype)))


def test_strided_rows_and_e4m3_results():
    announce('fp8 without exchange: strides')
    rng = np.random.default_rng(3)
    ai, bi, a, b = operands(rng, 40, 512, 384, False)
    one = torch.ones((), device='cuda')
    got = F8.matmul_f8_per_tensor(a[:, :256], b[:, 256:], one, torch.full((), 0.25, device='cuda'), output_dtype=torch.float8_e4m3fn)
    want = torch.from_numpy((ai[:, :256] @ bi[:, 256:].T).astype(np.float32) * 0.25).clamp(-448, 448).to(torch.float8_e4m3fn)
    assert np.array_equal(host(got.view(torch.uint8)), want.view(torch.uint8).numpy())


@pytest.mark.parametrize('m,k,n', [(33, 8192, 8192), (200, 8192, 4096), (512, 1024, 4096), (700, 2048, 2048)])
def test_narrow_tiles_beside(m, k, n):
    announce('fp8 narrow tiles', m, k, n)
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, False)
    one = torch.ones((), device='cuda')
    got = F8.matmul_f8_per_tensor(a, b, one, one, output_dtype=torch.float32)
    assert np.array_equal(host(got), ai.astype(np.float32) @ bi.T.astype(np.float32))


# Shapes that one-piece tiles of 32 rows, K whole, were chosen for: few column tiles then fetch the weight, one stage after the other, and from memory that
# is 10 to 30 % slower than tiles of 64 rows in two or three pieces, or strips (1 to 10 % from the cache, either way)
@pytest.mark.parametrize('m,k,n,scaled', [(308, 3024, 1856, False), (369, 3360, 1472, False), (277, 3680, 1856, False), (125, 5456, 7104, False), (337, 5760, 1824, False),
                                          (307, 2944, 1664, True), (155, 2944, 3456, True), (388, 3584, 1536, True)])
def test_weights_from_memory_not_in_one_piece(m, k, n, scaled):
    announce('fp8: not in one piece', m, k, n, scaled)
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, False)
    one = torch.ones((), device='cuda')
    if scaled:
        got = F8.matmul_f8_scaled(a, b, scale_a=torch.ones((k // 128, m), device='cuda'), scale_b=torch.ones((n // 128, k // 128), device='cuda'), output_dtype='float32')
    else:
        got = F8.matmul_f8_per_tensor(a, b, one, one, output_dtype=torch.float32)
    name, workgroups, _ = last_launch()
    one_piece = 8 * -(-(-(-m // 32) * -(-n // 128)) // 8)
    assert not (variant('MidF8', scaled, 2) in name and workgroups == one_piece), name
    assert np.array_equal(host(got), ai.astype(np.float32) @ bi.T.astype(np.float32))
