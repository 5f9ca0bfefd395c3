"""int8 matmuls on small row-major weights, which one workgroup per column strip computes over all of K: several row
tiles, waves without a step of K, K that ends inside a step, columns moved back into a row, rows of the weight at any alignment, a bias, strides; and sizes next to
those that take this kernel (its variants by name: test_gpu_strips.py). Small integers whose sums float16 holds: the results must be equal."""
import numpy as np
import pytest
import torch

from hidet_amd import ffi
from hidet_amd.graph.ops import quant
from gpu_util import announce, dev

pytestmark = pytest.mark.gpu


def _case(m, k, n):
    rng = np.random.default_rng(m + k + n)
    a, q = rng.integers(-2, 3, (m, k)).astype(np.float16), rng.integers(-2, 3, (k, n)).astype(np.int8)
    a *= rng.random((m, k)) < 0.5
    q[0, 0], q[k - 1, n - 1] = 127, -128
    exact = a.astype(np.float32) @ q.astype(np.float32)
    assert np.abs(exact).max() <= 2048
    return dev(a), dev(q), torch.from_numpy(exact)


@pytest.mark.parametrize('m', [1, 3, 16, 17, 33, 49, 64, 65, 130, 300])
@pytest.mark.parametrize('k,n', [(32, 4), (64, 6), (130, 34), (256, 256), (510, 1026), (1024, 64), (1024, 3000), (1118, 2050), (1500, 1006), (2048, 2048), (2046, 4102), (2050, 1024), (2514, 1030), (2560, 516), (2562, 520)])
def test_exact(m, k, n):
    announce('int8 small weight', m, k, n)
    a, q, exact = _case(m, k, n)
    one = torch.ones(n, dtype=torch.float16, device='cuda')
    assert torch.equal(quant.symmetric_quant_matmul(a, q, one).float().cpu(), exact)
    bias = (torch.arange(n, device='cuda') % 7).half()
    assert torch.equal(quant.symmetric_quant_matmul(a, q, one, bias).float().cpu(), (exact.half() + bias.cpu()).float())


@pytest.mark.parametrize('n', [5, 131, 1023])
def test_odd_columns_and_offsets_through_the_entry_point(n):
    announce('int8 small weight: odd N', n)
    m, k = 20, 384
    a, q, exact = _case(m, k, n)
    flat = torch.zeros(k * n + 3, dtype=torch.int8, device='cuda')
    wide = torch.zeros((m, k + 6), dtype=torch.float16, device='cuda')
    wide[:, :k] = a
    one = torch.ones(n, dtype=torch.float16, device='cuda')
    ws = ffi.workspace(a.device)
    for shift in range(4):
        w = flat[shift: shift + k * n]
        w.copy_(q.reshape(-1))
        c = torch.full((m, n), float('nan'), dtype=torch.float16, device='cuda')
        ffi.call('hidet_symmetric_quant_matmul_f16_i8', wide, w, one, c, m, k, n, k + 6, 0, ws, ws.numel(), ffi.current_stream(a.device))
        assert torch.equal(c.float().cpu(), exact)


def test_infinities_and_nan_stay_in_their_rows():
    announce('int8 small weight: infinity, NaN')
    a, q, exact = _case(18, 600, 512)
    a[3, 599], a[7, 0] = float('inf'), float('nan')
    q[599] = torch.where(q[599] == 0, torch.ones_like(q[599]), q[599])
    got = quant.symmetric_quant_matmul(a, q, torch.ones(512, dtype=torch.float16, device='cuda')).float().cpu()
    assert torch.isinf(got[3]).all() and torch.isnan(got[7]).all()
    keep = [i for i in range(18) if i not in (3, 7)]
    want = (a.float().cpu()[keep] @ q.float().cpu())
    assert torch.equal(got[keep], want)
