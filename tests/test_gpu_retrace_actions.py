"""Retrace with action counts outside {1, 2, 3, 4}: the action rows are reduced by a wave through
LDS, 64 rows at a time (rlk_ops.hpp reduce_actions), whole rows up to 18 actions (in batches of
5, 6, 9, 12 or 18 loads) and slices of 16 beyond."""
import numpy as np
import pytest
import torch

from _common import assert_close, make_inputs, run_api, run_oracle

pytestmark = pytest.mark.gpu


# rows of one wave, several rows per wave (whole and partial), several waves per row, rows of
# 1-3 steps (one step per lane), strided and look-back rows; the last wave of a row holding one
# step (257, 1025) or none (300 of 512, 1100 of 2048); the last three on both sides of the rule
# for one step per thread
@pytest.mark.parametrize("shape", [(3, 1), (5, 2), (70, 3), (1, 4), (9, 5), (33, 20), (65, 33), (40, 100),
                                   (300, 64), (7, 257), (5, 300), (3, 1025), (2, 1100), (2, 2049),
                                   (3, 5000), (300, 510), (1100, 130), (2100, 130)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("n_act", [3, 5, 6, 7, 9, 12, 13, 18, 19, 32, 33])
def test_retrace_any_action_count(n_act, shape, device):
    """Against the float64 oracle.  E_pi[Q'] sums n_act products of probabilities and N(0,1)
    values, so its float32 error stays that of the other terms: the suite's 1e-5."""
    inp, params = make_inputs("retrace", *shape, seed=n_act, n_act=n_act, p_trunc=0.02)
    params = dict(params, c_bar=0.9, rho_bar=0.8)
    got = run_api("retrace", inp, params, device)
    exp = run_oracle("retrace", inp, params)
    for g, e in zip(got, exp):
        assert_close(g.cpu().numpy(), e, 1e-5, 1e-5 * max(1.0, float(np.max(np.abs(e)))), f"A={n_act}{shape}")
    # bfloat16: the float32 result on the widened inputs, rounded (actions are integers)
    wide = {k: v if k == "actions" else torch.from_numpy(v).bfloat16().float().numpy() for k, v in inp.items()}
    want = [t.bfloat16() for t in run_api("retrace", wide, params, device)]
    got = run_api("retrace", wide, params, device, torch.bfloat16)
    for g, w in zip(got, want):
        assert torch.equal(g, w), f"bfloat16 A={n_act}{shape}"


@pytest.mark.parametrize("n_act", [3, 18, 40])
def test_retrace_action_outside_the_row(n_act, device):
    """An action outside [0, A) has probability 0, at a wave's edge as inside it."""
    inp, params = make_inputs("retrace", 6, 600, seed=2, n_act=n_act)
    acts = inp["actions"].copy()
    acts[:, ::5] = -1
    acts[:, 256::256] = n_act
    acts[:, 3::7] = n_act + 1000
    got = run_api("retrace", dict(inp, actions=acts), params, device)
    pi = inp["action_probs_target"].copy()
    outside = (acts < 0) | (acts >= n_act)
    # the same recurrence with a taken probability of 0: mu = inf makes the ratio 0
    mu = np.where(outside, np.float32(np.inf), inp["action_probs_behavior"])
    exp = run_oracle("retrace", dict(inp, action_probs_target=pi, action_probs_behavior=mu,
                                     actions=np.where(outside, 0, acts)), params)
    for g, e in zip(got, exp):
        assert_close(g.cpu().numpy(), e, 1e-5, 1e-5 * max(1.0, float(np.max(np.abs(e)))), f"A={n_act}")
