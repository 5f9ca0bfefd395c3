"""A launch of 2^32 threads or more along one axis would run in part only: it has to be an error, raised on the host before anything runs."""
import pytest

from hidet_amd import ffi


@pytest.mark.parametrize('outer,reduce,inner', [(1, 32 * 4096, 1 << 20), (1, 1 << 34, 128), (2, 32 * 4097, (1 << 20) + 1)])
def test_a_grid_beyond_the_limit_is_an_error(outer, reduce, inner):
    with pytest.raises(ffi.BackendException, match='too large for one launch'):
        ffi.call('hidet_symmetric_dequantize', 4096, 4096, 4096, outer, reduce, inner, ffi.I8, ffi.F32, 0)
