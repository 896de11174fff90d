"""The extension module of csrc/torch: used with the torch that it was built for alone, and no condition of a build."""
import os
import sys
import warnings

import pytest
import torch

from kubernetes_cloud_amd.ops import _lib

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tools"))
import build_ext  # noqa: E402


@pytest.mark.skipif(not os.path.exists(os.path.join(_lib.LIB_DIR, "kca_torch.so")) or not _lib.available(), reason="not built")
def test_another_torch(monkeypatch):
    monkeypatch.setattr(_lib, "_torch_ext", [])
    monkeypatch.setattr(_lib.torch, "__version__", "0.0.1")
    with pytest.warns(UserWarning, match="built for torch"):
        assert _lib.torch_ext() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.torch_ext() is None  # said once
    monkeypatch.undo()
    monkeypatch.setattr(_lib, "_torch_ext", [])
    assert _lib.torch_ext().torch == torch.__version__


@pytest.mark.skipif(not os.path.exists(os.path.join(_lib.LIB_DIR, "kca_torch.so")) or not _lib.available(), reason="not built")
def test_a_library_without_prompt_kernels(monkeypatch):
    """A library of a few sources: attention stays in the module, a prompt layer's operators go to Python."""
    class Partial:
        def __getattr__(self, n):
            if n == "kca_rope_append":
                raise AttributeError(n)
            return getattr(lib, n)
    lib = _lib._load()
    with torch.no_grad(), monkeypatch.context() as mp:
        mp.setattr(_lib, "_torch_ext", [])
        mp.setattr(_lib, "_load", lambda: Partial())
        assert _lib.torch_ext() is not None and _lib.plain_ext() is None
    with torch.no_grad(), monkeypatch.context() as mp:
        mp.setattr(_lib, "_torch_ext", [])
        assert _lib.plain_ext() is _lib.torch_ext() is not None
    assert _lib.plain_ext() is None  # gradients


def test_a_build_without_it(monkeypatch, capsys):
    monkeypatch.setattr(build_ext, "build_kernels", lambda *a, debug=False, **k: "debug" if debug else "kernels")
    monkeypatch.setattr(build_ext, "build_host", lambda *a: "host")

    def no_headers(*a):
        raise RuntimeError("compile failed")
    monkeypatch.setattr(build_ext, "build_torch", no_headers)
    assert build_ext.build_all() == ("kernels", "host", None, "debug")
    assert "kca_torch.so not built" in capsys.readouterr().err
