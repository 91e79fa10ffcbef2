"""The Python extension is tied to the torch and Python it was compiled against."""
import pytest


@pytest.fixture
def native(monkeypatch):
  from cache_dit_amd import _native
  if not _native.is_built():
    pytest.skip("libcdit_hip.so not built")
  monkeypatch.setattr(_native, "_host", None)
  return _native


def test_extension_of_another_torch_is_refused(native, monkeypatch, tmp_path):
  """Before it is loaded, with a message that says what to do."""
  import torch
  with open(native.HOST_PATH, "rb") as f:
    built = f.read()
  version = f"torch {torch.__version__}".encode()
  assert version in built
  other = tmp_path / "_cdit_host.so"
  other.write_bytes(built.replace(version, b"torch 0" + version[7:]))
  monkeypatch.setattr(native, "HOST_PATH", str(other))
  assert not native.is_built()
  with pytest.raises(native.CditNativeError, match="rebuild"):
    native.host()
  assert native._host is None


def test_extension_of_this_torch_is_taken(native):
  assert native.host() is native.host()
