"""The 256 x 128 FP8 tiles at the sizes where their loops can go wrong: one, two and three k blocks (the ring is three deep), more
than 64 (column factors come 64 at a time), full, part-filled and short row tiles, K ranges. Integer-valued codes and
scales whose sums stay below 2^24: exact in float32, so the results must be equal."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from hidet_amd.graph.ops.matmul import matmul_f8 as F8
from gpu_util import announce, dev, host

pytestmark = pytest.mark.gpu


def operands(rng, m, k, n, e5m2):
    ai, bi = rng.integers(-4, 5, (m, k)), rng.integers(-4, 5, (n, k))
    enc, dtype = (O.e5m2_encode, torch.float8_e5m2) if e5m2 else (O.e4m3_encode, torch.float8_e4m3fn)
    return ai, bi, dev(enc(ai.astype(np.float32))).view(dtype), dev(enc(bi.astype(np.float32))).view(dtype)


# e5m2 operands take these tiles from 17 rows on, e4m3 above 1024
@pytest.mark.parametrize('m,k,n,e5m2', [(1025, 128, 128, False), (1280, 256, 384, False), (1217, 384, 256, False), (1300, 8192 + 128, 128, False),
                                        (1216, 128 * 130, 128, False), (17, 128, 128, True), (65, 8192 + 256, 128, True),
                                        (129, 128 * 66, 256, True), (193, 640, 128, True), (256, 128 * 65, 128, True),
                                        # 129 to 192 rows of the last tile, which is computed as a full one; with K ranges and without
                                        (1153, 128, 256, False), (1180, 128 * 9, 3072, False), (2200, 7168, 1536, False), (192, 1024, 256, True)])
def test_block_scaled(m, k, n, e5m2):
    announce('block-scaled tiles', m, k, n, e5m2)
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, e5m2)
    sa = rng.integers(1, 5, (k // 128, m)).astype(np.float32)
    sb = rng.integers(1, 5, (n // 128, k // 128)).astype(np.float32)
    got = F8.matmul_f8_scaled(a, b, scale_a=dev(sa), scale_b=dev(sb), output_dtype='float32')
    exact = (ai * np.repeat(sa.T, 128, axis=1)).astype(np.float64) @ (bi * np.repeat(np.repeat(sb, 128, axis=0), 128, axis=1)).T.astype(np.float64)
    assert np.abs(exact).max() < 2 ** 24
    assert np.array_equal(host(got), exact.astype(np.float32))


@pytest.mark.parametrize('m,k,n', [(1025, 128, 132), (1280, 256, 1000), (2048, 384, 1024), (1217, 8320, 260), (1153, 128, 260), (1200, 1152, 1000), (2190, 4096, 1536)])
def test_per_tensor(m, k, n):
    announce('per-tensor tiles', m, k, n)
    rng = np.random.default_rng(m + k + n)
    ai, bi, a, b = operands(rng, m, k, n, False)
    one = torch.ones((), device='cuda')
    got = F8.matmul_f8_per_tensor(a, b, one, one, output_dtype=torch.float16)
    exact = ai.astype(np.float64) @ bi.T.astype(np.float64)
    assert np.array_equal(host(got), exact.astype(np.float32).astype(np.float16))
