"""int8 matmuls of 17 to 64 rows on small K-contiguous weights, and of any number where K is no multiple of 128 (above 64, through the entry point alone, of 64), which one workgroup per column strip computes over
all of K: waves without a step of K, K that ends inside a step, rows and columns past the end, a bias, strided activations; and shapes that stay with the narrow tiles (the
variants of the kernel by name: test_gpu_strips.py). Small integers whose sums float16 holds: the results must be equal."""
import numpy as np
import pytest
import torch

from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev, last_launch

pytestmark = pytest.mark.gpu


def _case(m, k, n):
    rng = np.random.default_rng(m + k + n)
    a, q = rng.integers(-2, 3, (m, k)).astype(np.float16), rng.integers(-2, 3, (k, n)).astype(np.int8)
    a[:, 3:] *= (rng.random(k - 3) < 0.5)
    q[0, 0], q[k - 1, n - 1] = 127, -128
    exact = a.astype(np.float32) @ q.astype(np.float32)
    assert np.abs(exact).max() <= 2048
    return dev(a), quant.to_decode_layout(dev(q)), torch.from_numpy(exact)


@pytest.mark.parametrize('m', [1, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize('k,n', [(16, 8), (128, 20), (1024, 1024), (1040, 2052), (1088, 4096), (2048, 6144), (4096, 1000), (4096, 4096), (3008, 11008)])
def test_exact(m, k, n):
    announce('int8 K-contiguous', m, k, n)
    a, w, exact = _case(m, k, n)
    one = torch.ones(n, dtype=torch.float16, device='cuda')
    assert torch.equal(quant.symmetric_quant_matmul(a, w, one).float().cpu(), exact)
    bias = (torch.arange(n, device='cuda') % 7).half()
    assert torch.equal(quant.symmetric_quant_matmul(a, w, one, bias).float().cpu(), (exact.half() + bias.cpu()).float())


def test_random_against_float64():
    announce('int8 K-contiguous: random')
    g = torch.Generator(device='cuda').manual_seed(1)
    for m, k, n in [(24, 2048, 2048), (64, 1536, 3072)]:
        w, scale = quant.symmetric_quantize(torch.randn((k, n), generator=g, device='cuda') * 0.02, 'int8', dims=0)
        x, scale = torch.randn((m, k), generator=g, device='cuda').half(), scale.half()
        want = (x.double() @ w.double()) * scale.double()
        got = quant.symmetric_quant_matmul(x, quant.to_decode_layout(w), scale).double()
        assert 'skinny_w8a16_nk_tall_kernel' in last_launch()[0]
        # float32 sums of k products: at most 2^-24 log2(k) of the sum of their magnitudes each way, and half a unit of float16
        bound = (x.double().abs() @ w.double().abs()) * scale.double() * 2.0 ** -24 * (k / 128 + 12) + want.abs() * 2.0 ** -11 + 2.0 ** -24
        assert ((got - want).abs() <= bound).all()


def test_strided_activations():
    announce('int8 K-contiguous: strides')
    a, w, exact = _case(40, 1024, 512)
    one = torch.ones(512, dtype=torch.float16, device='cuda')
    for pad in (8, 2, 1):  # rows of 16-byte pieces, and rows that are not
        wide = torch.zeros((40, 1024 + pad), dtype=torch.float16, device='cuda')
        wide[:, :1024] = a
        assert torch.equal(quant.symmetric_quant_matmul(wide[:, :1024], w, one).float().cpu(), exact)


@pytest.mark.parametrize('m', [65, 130, 201])
def test_more_rows_of_k_off_the_stages_through_the_entry_point(m):
    announce('int8 K-contiguous: more rows', m)
    a, w, exact = _case(m, 1040, 516)
    one, c = torch.ones(516, dtype=torch.float16, device='cuda'), torch.empty((m, 516), dtype=torch.float16, device='cuda')
    ffi.call('hidet_symmetric_quant_matmul_f16_i8_nk', a, w.T.contiguous(), one, c, m, 1040, 516, 1040, 1040, None, 0, ffi.current_stream(a.device))
    assert torch.equal(c.float().cpu(), exact)
    assert 'skinny_w8a16_nk_tall_kernel' in last_launch()[0]
