"""What a call of the fused min / max form derives from shapes and options (mi355x_qdq._call_of), on
the CPU."""
import sys
import warnings
from pathlib import Path

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "rx-met_amd"))
import mi355x_qdq as Q  # noqa: E402
import rxmet_lib  # noqa: E402


def _call(x, mn):
    return Q._call_of(x, mn, -8, 7, False, 1e-8, 0.0, None, 0.0)


def test_traced_calls_share_the_plan_of_their_shape():
    """Under torch.jit.trace the sizes of a tensor are tensors; the plans are keyed by their values,
    so traces of one shape, and the call outside, meet one plan and keep no traced tensor."""

    class Traced(torch.nn.Module):
        def forward(self, x):
            seen.append(_call(x, mn))
            return x + 1

    seen, mn = [], torch.zeros(37, 1)
    Q._minmax_call.cache_clear()
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", torch.jit.TracerWarning)
        for _ in range(2):
            torch.jit.trace(Traced(), torch.zeros(37, 53), check_trace=False)
    seen.append(_call(torch.zeros(37, 53), mn))
    assert Q._minmax_call.cache_info().currsize == 1
    assert seen[0] is not None and all(c is seen[0] for c in seen)


def test_without_the_torch_module(monkeypatch):
    """Where rxmet_torch cannot be imported the calls warn once and keep the Python Function."""
    monkeypatch.setattr(rxmet_lib, "_torch_ext", None)
    monkeypatch.setitem(sys.modules, "rxmet_torch", None)  # its import raises ImportError
    Q._minmax_call.cache_clear()
    mn = torch.zeros(5, 1)
    try:
        with pytest.warns(UserWarning, match="rxmet_torch"):
            call = _call(torch.zeros(5, 8), mn)
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            other = _call(torch.zeros(5, 9), mn)
        for c in (call, other):
            assert c.plan is not None and c.native is None
    finally:
        Q._minmax_call.cache_clear()  # plans without a native node
