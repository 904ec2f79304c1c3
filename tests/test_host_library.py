"""A native call path that is missing or was compiled against another torch says
what to do, as the missing kernel library does."""
import pytest

from bozo_amd import _lib as L


@pytest.mark.parametrize("content", [None, b"", b"\x7fELF not one"])
def test_unusable_call_path_names_the_build(tmp_path, monkeypatch, content):
    path = tmp_path / "_host.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(L, "HOST_PATH", str(path))
    monkeypatch.setattr(L, "_host", None)
    with pytest.raises(L.TensionError, match="python -m bozo_amd.build") as e:
        L.host()
    assert str(path) in str(e.value)


def test_built_call_path_loads():
    assert L.host() is L.host()
