"""A call of more rows times columns than the threads of one launch take, at 512 per workgroup and 64 x 32 results: computed in ranges of rows. Small integers: equal at
sampled rows of both."""
import pytest
import torch

from hidet_amd import ffi
from gpu_util import announce

pytestmark = pytest.mark.gpu


def test_int8_k_contiguous_off_the_steps():
    m, k, n = 65536 + 40, 80, 1 << 18
    announce('K-contiguous, large launch', m, k, n)
    g = torch.Generator(device='cuda').manual_seed(1)
    a = torch.randint(-2, 3, (m, k), generator=g, device='cuda').half()
    w = torch.randint(-2, 3, (n, k), generator=g, device='cuda', dtype=torch.int8)
    one, c = torch.ones(n, dtype=torch.float16, device='cuda'), torch.empty((m, n), dtype=torch.float16, device='cuda')
    ffi.call('hidet_symmetric_quant_matmul_f16_i8_nk', a, w, one, c, m, k, n, k, k, None, 0, ffi.current_stream(a.device))
    rows = torch.tensor([0, 63, 64, 8175, 8176, 8177, m // 2, m - 40, m - 1], device='cuda')
    assert torch.equal(c[rows].float(), a[rows].float() @ w.float().T.contiguous())
    del c
    torch.cuda.empty_cache()
