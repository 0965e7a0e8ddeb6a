"""The native call module leaves everything but plain device tensors of the documented types to the Python
wrappers: it returns None, raises nothing and launches nothing."""

import importlib.util

import pytest
import torch

from q4llm._lib import PKG, native_calls

mod = native_calls()


def test_built():
    assert mod is not None and all(hasattr(mod, n) for n in ("gemv", "linear", "attn", "gemm"))


@pytest.mark.parametrize("lacks", ["torch", "headers"])
def test_build_without_torch(monkeypatch, tmp_path, lacks):
    """The library and the native runner need no torch: the build leaves the module out where there is no
    torch to build it for, and takes an older one away, which could not match the new library."""
    spec = importlib.util.spec_from_file_location("q4_build", PKG / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    fake = importlib.util.spec_from_loader("torch", None, is_package=True)
    fake.submodule_search_locations.append(str(tmp_path))
    monkeypatch.setattr(importlib.util, "find_spec", lambda name: None if lacks == "torch" else fake)
    monkeypatch.setattr(build, "LIB", tmp_path)
    (tmp_path / "_q4torch.so").write_bytes(b"old")
    assert build.build_torch_module() is None
    assert not (tmp_path / "_q4torch.so").exists()


@pytest.mark.parametrize("bad", [None, 1, "x", torch.zeros(2, 4, dtype=torch.int32), torch.zeros(0), object()])
def test_leaves_the_rest_to_python(bad):
    qw, sc, x = torch.zeros(8, 8, dtype=torch.int32), torch.zeros(8, 2, dtype=torch.float16), torch.zeros(1, 64)
    for args in ([bad, sc, x[0], 32, 0, None, None], [qw, bad, x[0], 32, 0, None, None], [qw, sc, bad, 32, 0, None, None],
                 [qw, sc, x[0], bad, 0, None, None], [qw, sc, x[0], 1 << 70, 0, None, None], [qw, sc]):
        assert mod.gemv(*args) is None
    assert mod.linear(qw, sc, x, 32, bad, True) is None and mod.linear(bad, sc, x, 32, None, False) is None
    assert mod.attn(bad, x, x, 4, x, 0.5, None) is None and mod.gemm(bad, x, None) is None and mod.gemm() is None
