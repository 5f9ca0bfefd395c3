"""Without a native front that can be loaded the operators keep their Python path."""
import pytest

from hidet_amd import ffi


@pytest.mark.parametrize('content', [None, b'no shared object'])
def test_a_front_that_cannot_be_loaded_handles_nothing(tmp_path, monkeypatch, content):
    path = tmp_path / '_front.so'
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(ffi, 'FRONT_PATH', str(path))
    monkeypatch.setattr(ffi, '_FRONT', None)
    with pytest.warns(RuntimeWarning, match='cannot be loaded'):
        front = ffi.front()
    assert front.w8a16(None, None, None, None) is None and front.quantize(None, None, 0) is None
    assert ffi.front() is front  # looked for once
