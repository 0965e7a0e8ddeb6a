"""The native call module leaves everything but plain device tensors of the documented types to the Python
wrappers: it returns None, raises nothing and launches nothing."""

import pytest
import torch

from q4llm._lib import native_calls

mod = native_calls()


def test_built():
    assert mod is not None and all(hasattr(mod, n) for n in ("gemv", "linear", "attn", "gemm"))


@pytest.mark.parametrize("bad", [None, 1, "x", torch.zeros(2, 4, dtype=torch.int32), torch.zeros(0), object()])
def test_leaves_the_rest_to_python(bad):
    qw, sc, x = torch.zeros(8, 8, dtype=torch.int32), torch.zeros(8, 2, dtype=torch.float16), torch.zeros(1, 64)
    for args in ([bad, sc, x[0], 32, 0, None, None], [qw, bad, x[0], 32, 0, None, None], [qw, sc, bad, 32, 0, None, None],
                 [qw, sc, x[0], bad, 0, None, None], [qw, sc, x[0], 1 << 70, 0, None, None], [qw, sc]):
        assert mod.gemv(*args) is None
    assert mod.linear(qw, sc, x, 32, bad, True) is None and mod.linear(bad, sc, x, 32, None, False) is None
    assert mod.attn(bad, x, x, 4, x, 0.5, None) is None and mod.gemm(bad, x, None) is None and mod.gemm() is None
