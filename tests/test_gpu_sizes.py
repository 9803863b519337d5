"""GPU parity at the sizes where the kernels' per-thread and per-wave splits
end: the smallest vectors, remainders past one element group per thread, odd
chunk counts.  Against the CPU oracle, at the repository's bar (max-abs-rel
2e-2, barrier tensor equal)."""

import pytest

from llama_harness import LlamaCase
from megakernels_amd.latency.synthetic import LlamaConfig

pytestmark = pytest.mark.gpu
TOL = 2e-2


def _check(case, name):
    err = case.errors()
    print(f"[{name}] " + " ".join(f"{k} {v:.2e}" for k, v in err.items()), flush=True)
    for k, v in err.items():
        assert v <= TOL, f"{name} {k}: max-abs-rel {v:.3e}"
    assert case.barriers_equal(), "barrier tensor differs from the oracle's"


@pytest.mark.parametrize("hidden,heads,kv_heads", [(512, 8, 2), (4096, 32, 16), (4608, 36, 9)])
def test_dense_hidden_sizes(hidden, heads, kv_heads):
    """The norm keeps 8 elements of the hidden state per thread: one wave of
    it, exactly one group per thread, and a second group for some threads."""
    case = LlamaCase(LlamaConfig(1, hidden, 1024, heads, kv_heads, 64), seed=3, prefill=40, steps=1)
    case.step(5)
    _check(case, f"dense H {hidden}")
