"""The launch layer's extension module where it cannot be used: missing, built for
another ABI or another PyTorch.  Calls then go the Python way, with a warning."""

from __future__ import annotations

import pytest
import torch

from SSA import _lib


@pytest.fixture
def reload(monkeypatch):
    """Forgets the loaded module for the test; its path and the library can be replaced."""
    monkeypatch.setattr(_lib, "_native", None)
    return monkeypatch


def _is_python_path(mod):
    x = torch.zeros(1, 2, 32, 64)
    return (isinstance(mod, _lib.PythonPath) and mod.fwd(x, x, x, 0.1, x, x, True, 0, 0) is None
            and mod.bwd() is None and mod.headroom(0) is None)


def test_missing(reload, tmp_path):
    from SSA import ssa_decode_num_splits

    reload.setattr(_lib, "NATIVE_PATH", tmp_path / "_ssa_native.so")
    with pytest.warns(RuntimeWarning, match="not been built"):
        mod = _lib.native()
    assert _is_python_path(mod) and _lib.native() is mod  # one warning, not one a call
    # the library's own split rule
    assert ssa_decode_num_splits(1, 16, 16, 4096) == _lib.lib().ssa_decode_num_splits(1, 16, 16, 4096, 0)


def test_not_loadable(reload, tmp_path):
    (tmp_path / "_ssa_native.so").write_bytes(b"not a shared object")
    reload.setattr(_lib, "NATIVE_PATH", tmp_path / "_ssa_native.so")
    with pytest.warns(RuntimeWarning):
        assert _is_python_path(_lib.native())


def test_other_abi(reload):
    real = _lib.lib()

    class Newer:
        def __getattr__(self, name):
            return (lambda: _lib.ABI_VERSION + 1) if name == "ssa_abi_version" else getattr(real, name)

    reload.setattr(_lib, "lib", lambda: Newer())
    with pytest.warns(RuntimeWarning, match="ABI version"):
        assert _is_python_path(_lib.native())


def test_other_pytorch(reload):
    reload.setattr(torch, "__version__", "1.0.0")
    with pytest.warns(RuntimeWarning, match="PyTorch"):
        assert _is_python_path(_lib.native())


def test_present():
    assert not isinstance(_lib.native(), _lib.PythonPath)
    assert _lib.native().ABI_VERSION == _lib.ABI_VERSION
