"""The buffers kept per stream (look-back workspaces, the one-launch normalised GAE's) are ordinary
tensors: first used under torch.inference_mode(), they are zero-filled again at the call limit
outside it."""
import ctypes

import pytest
import torch

from _common import assert_close, make_inputs, run_api, run_oracle, suite_atol

pytestmark = pytest.mark.gpu


def _fresh_stream():
    """A stream that no earlier call has used (torch's own come from a pool)."""
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    return torch.cuda.ExternalStream(s.value)


@pytest.mark.parametrize("path", ["fast", "python"])
@pytest.mark.parametrize("op,shape", [("gae_normalized", (1024, 128)), ("gae", (3, 40000))],
                         ids=["normalised", "lookback"])
def test_buffers_made_under_inference_mode(op, shape, path, device, monkeypatch):
    from rl_triton import _native
    if path == "fast":
        monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    monkeypatch.setattr(_native, "WORKSPACE_MAX_CALLS", 3)
    inp, params = make_inputs(op, *shape, seed=1, boot="row")
    want = run_oracle(op, inp, params)
    prev = _native.fast.set_workspace_max_calls(3)
    clears = lambda: _native._ws_clears + _native.fast.workspace_clears() + _native.fast.sync_clears()  # noqa: E731
    launched, cleared = _native.fast.launched(), clears()
    try:
        with torch.cuda.stream(_fresh_stream()):
            with torch.inference_mode():
                run_api(op, inp, params, device)
            for _ in range(7):
                got = run_api(op, inp, params, device)
            torch.cuda.synchronize()
    finally:
        _native.fast.set_workspace_max_calls(prev)
    if path == "fast":
        assert _native.fast.launched() - launched == 8
    if path == "fast" or op == "gae":  # (normalised GAE of short rows keeps nothing on the Python path)
        assert clears() - cleared == 2
    for g, w in zip(got, want):
        assert_close(g.cpu().numpy(), w, 1e-5, 4 * suite_atol("gae", inp, w, shape[1]), op)
