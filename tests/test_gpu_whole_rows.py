"""Rows of more than 2048 steps held whole by one workgroup (whole_row in csrc/rlk_launch.hpp): one,
two or four 4-step segments per thread, as many waves as the row needs."""
import numpy as np
import pytest
import torch

from _common import OUTPUTS, assert_close, make_inputs, run_api, run_oracle, suite_atol

pytestmark = pytest.mark.gpu

OPS = ["gae", "gae_masked", "gae_normalized", "gae_normalized_masked", "vtrace", "retrace", "lambda_returns",
       "discounted_returns", "eligibility_traces", "prefix_sum", "backward_scan", "forward_scan"]


# the ends of each segment count's range, one step into a wave, one short of a whole wave; the
# four-segment ones with a row for half the CUs of a 256-CU GPU, and one row fewer
@pytest.mark.parametrize("shape", [(3, 2049), (2, 2052), (5, 2304), (2, 2305), (3, 4095), (2, 4096), (3, 4097),
                                   (2, 4100), (300, 4609), (257, 8191), (2, 8192), (127, 8193), (128, 8193),
                                   (129, 8196), (130, 9217), (128, 9002), (128, 16383), (128, 16384)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("op", OPS)
def test_whole_rows(op, shape, device):
    if op in ("prefix_sum", "gae_masked", "gae_normalized_masked") and shape[0] * shape[1] > 1 << 21 and shape[1] % 4:
        pytest.skip("the oracle is slow here; the smaller element-aligned shapes cover each segment count")
    kw = {"p_done": 1e-2} if op in ("prefix_sum", "eligibility_traces") else {}
    trunc = 0.01 if op in ("gae", "vtrace", "gae_normalized") else 0.0
    inp, params = make_inputs(op, *shape, seed=shape[0] + shape[1], p_trunc=trunc,
                              boot="full" if trunc else "none", **kw)
    got = run_api(op, inp, params, device)
    exp = run_oracle(op, inp, params)
    base = op.replace("_masked", "").replace("_normalized", "")
    for name, g, e in zip(OUTPUTS[op], got, exp):
        # the suite's long-row tolerance; normalised advantages carry it over their std (above 1)
        assert_close(g.cpu().numpy(), e, 1e-5, 4 * suite_atol(base, inp, e, shape[1]), f"{op}{shape}:{name}")
    if "normalized" in op:
        return
    wide = {k: v if v is None or k == "actions" else torch.from_numpy(np.asarray(v)).bfloat16().float().numpy()
            for k, v in inp.items()}
    half = run_api(op, wide, params, device, torch.bfloat16)
    for name, h, w in zip(OUTPUTS[op], half, run_api(op, wide, params, device)):
        assert torch.equal(h, w.bfloat16()), f"{op}{shape}:{name} bfloat16"


@pytest.mark.parametrize("op", ["discounted_returns", "prefix_sum"])
@pytest.mark.parametrize("shape", [(2, 2500), (2, 8000), (128, 9000)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_non_finite_input_spreads_as_in_the_loop(op, shape, device):
    """One workgroup per row: an inf makes every later step in scan order non-finite, resets or
    not (0 * inf is nan), as the sequential loop does."""
    inp, params = make_inputs(op, *shape, seed=31, p_term=0.0, p_done=0.0)
    inp["terminateds" if op == "discounted_returns" else "dones"][:, 150::300] = 1.0
    inp["rewards" if op == "discounted_returns" else "inputs"][:, shape[1] // 2] = np.inf
    exp = run_oracle(op, inp, params)[0]
    got = run_api(op, inp, params, device)[0].cpu().numpy()
    assert np.array_equal(np.isfinite(got), np.isfinite(exp))
