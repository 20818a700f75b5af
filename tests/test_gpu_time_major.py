"""Public calls on transposed views of [T, E] buffers: read in place by the time-major kernels
(csrc/rlk_columns.hpp) for rows of up to 2048 steps, copied to rows otherwise."""
import numpy as np
import pytest
import torch

from _common import OUTPUTS, assert_close, make_inputs, run_oracle

pytestmark = pytest.mark.gpu


def _columns(inp, device, dtype=torch.float32, ld=None, drop=()):
    """The case's [E, T] and [E, T, A] arrays as transposed views of [T, ld >= E] buffers."""
    out = {}
    for k, v in inp.items():
        t = None if v is None else torch.as_tensor(np.asarray(v))
        if t is None:
            out[k] = None
            continue
        if t.is_floating_point():
            t = t.to(dtype)
        t = t.to(device)
        if t.dim() > 1 and k not in drop:
            n = t.shape[0]
            buf = torch.zeros((t.shape[1], ld or n, *t.shape[2:]), dtype=t.dtype, device=device)
            buf[:, :n].copy_(t.transpose(0, 1))
            t = buf[:, :n].transpose(0, 1)
        out[k] = t
    return out


def _call(op, d, params):
    import rl_triton
    g = d.get
    boots = dict(bootstrap_values=g("bootstrap_values"))
    if op.startswith("gae"):
        fn = rl_triton.compute_gae_normalized if "normalized" in op else rl_triton.compute_gae
        res = fn(g("rewards"), g("values"), g("terminateds"), g("truncateds"), **boots,
                 last_value=g("last_value"), mask=g("mask"), **params)
    elif op == "vtrace":
        res = rl_triton.compute_vtrace(g("log_pi_target"), g("log_pi_behavior"), g("values"), g("rewards"),
                                       g("terminateds"), g("truncateds"), **boots, last_value=g("last_value"),
                                       **params)
    elif op == "retrace":
        res = rl_triton.compute_retrace(g("action_probs_target"), g("action_probs_behavior"), g("q_values"),
                                        g("next_q_values_all"), g("actions"), g("rewards"), g("terminateds"),
                                        g("truncateds"), **params)
    elif op == "lambda_returns":
        res = rl_triton.compute_lambda_returns(g("rewards"), g("next_values"), g("terminateds"), g("truncateds"),
                                               **boots, **params)
    elif op == "discounted_returns":
        res = rl_triton.compute_discounted_returns(g("rewards"), g("terminateds"), g("truncateds"), **boots,
                                                   **params)
    elif op == "eligibility_traces":
        res = rl_triton.compute_eligibility_traces(g("gradients"), g("dones"), params["gamma"], params["lambda_"],
                                                   seed_values=g("seed_values"))
    else:
        res = rl_triton.compute_episodic_prefix_sum(g("inputs"), g("dones"), seed_values=g("seed_values"),
                                                    boundary=params.get("boundary", "ends_at"))
    return res if isinstance(res, tuple) else (res,)


@pytest.fixture
def no_flags(monkeypatch):
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)


# one chunk to several passes (256 steps each), partial chunks and passes, column groups
# of 1 to 16 environments, several groups per workgroup
SHAPES = [(2, 2), (5, 3), (16, 5), (17, 16), (31, 17), (33, 33), (100, 64), (15, 100), (64, 128), (129, 130),
          (40, 256), (7, 257), (300, 250), (20, 600), (3, 2048)]
OPS = ["gae", "gae_masked", "gae_normalized", "gae_normalized_masked", "vtrace", "retrace", "lambda_returns",
       "discounted_returns", "eligibility_traces", "prefix_sum"]


def _inputs(op, shape, boot, trunc, n_act=4):
    inp, params = make_inputs(op, *shape, seed=shape[0] + shape[1], p_trunc=trunc, boot=boot, n_act=n_act)
    if op in ("lambda_returns", "discounted_returns"):
        inp.pop("last_value", None)
    if inp.get("mask") is not None and inp["mask"].sum() < 2:  # the std of fewer steps is nan
        inp["mask"][:] = 1
    return inp, params


def _check(op, inp, params, device, what, ld=None):
    from rl_triton import _native
    before = _native.fast.launched()
    got = _call(op, _columns(inp, device, ld=ld), params)
    assert _native.fast.launched() == before + 1, f"{what}: not taken by the fast path"
    exp = run_oracle(op, inp, params)
    scale = max(1.0, *(float(np.max(np.abs(e))) for e in exp))
    for name, g, e in zip(OUTPUTS[op], got, exp):
        assert g.is_contiguous() and tuple(g.shape) == e.shape
        # the suite's 1e-5, of the largest result (the normalised advantages divide by a std
        # that can be below 1)
        assert_close(g.cpu().numpy(), e, 1e-5, (4e-5 if "normalized" in op else 1e-5) * scale, f"{what}:{name}")
    # bfloat16: the float32 result on the widened inputs, rounded; the advantages that
    # compute_gae_normalized normalises are rounded before that too (by 2^-8 of them at most, over
    # their std)
    wide = {k: v if v is None or k == "actions" else torch.from_numpy(np.asarray(v)).bfloat16().float().numpy()
            for k, v in inp.items()}
    want = _call(op, _columns(wide, device, ld=ld), params)
    half = _call(op, _columns(wide, device, torch.bfloat16, ld=ld), params)
    atol = 1e-5 * scale
    if "normalized" in op:
        a = want[1].cpu().numpy() - wide["values"]
        kept = a if wide.get("mask") is None else a[wide["mask"] != 0]
        atol += 1.01 * 2.0 ** -8 * float(np.max(np.abs(a))) / float(np.std(kept, ddof=1))
    for name, h, w in zip(OUTPUTS[op], half, want):
        assert h.dtype == torch.bfloat16
        if "normalized" not in op:
            assert torch.equal(h, w.bfloat16()), f"{what}:{name} bfloat16"
        assert_close(h.float().cpu().numpy(), w.cpu().numpy(), 2.0 ** -8, atol, f"{what}:{name} bfloat16")


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("boot,trunc", [("none", 0.0), ("row", 0.0), ("full", 0.05)])
def test_time_major(op, shape, boot, trunc, device, no_flags):
    inp, params = _inputs(op, shape, boot, trunc)
    _check(op, inp, params, device, f"{op}{shape} boot={boot}")


@pytest.mark.parametrize("n_act", [1, 2, 3, 5, 6, 9, 12, 18, 19, 40])
@pytest.mark.parametrize("shape", [(2, 3), (17, 33), (40, 300)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_time_major_action_counts(n_act, shape, device, no_flags):
    inp, params = _inputs("retrace", shape, "none", 0.02, n_act)
    _check("retrace", inp, params, device, f"A={n_act}{shape}")


def test_time_major_slices(device, no_flags):
    """Views into wider buffers (some of a collector's environments; all but the last step)."""
    for op in ("gae", "retrace", "prefix_sum"):
        inp, params = _inputs(op, (37, 70), "row", 0.0)
        _check(op, inp, params, device, f"{op} ld=50", ld=50)


def test_time_major_starts_at(device, no_flags):
    inp, params = _inputs("prefix_sum", (33, 270), "row", 0.0)
    _check("prefix_sum", inp, {"boundary": "starts_at"}, device, "starts_at")


@pytest.mark.parametrize("op", OPS)
def test_time_major_mixed_layouts_take_the_general_path(op, device, no_flags):
    """Arrays of different layouts or strides, and rows above 2048 steps: the same results by
    copies."""
    from rl_triton import _native
    shapes = [((40, 60), dict(drop=("terminateds", "dones"))), ((5, 2049), {})]
    for shape, kw in shapes + ([((40, 600), {})] if op == "retrace" else []):
        # (Retrace, 40 environments: more than four actions and more than 512 steps)
        inp, params = _inputs(op, shape, "none", 0.0, 4 if shape[1] != 600 else 5)
        d = _columns(inp, device, **kw)
        before = _native.fast.launched()
        got = _call(op, d, params)
        if shape[1] <= 2048:
            assert _native.fast.launched() == before
        want = _call(op, {k: v if v is None else v.contiguous() for k, v in d.items()}, params)
        for g, w in zip(got, want):
            assert torch.equal(g, w), f"{op}{shape}"


def test_time_major_negative_views_and_capture(device, no_flags):
    import rl_triton
    x = torch.randn(64, 48, device=device)
    neg = torch._neg_view(x).t()
    got = rl_triton.compute_gae(neg, neg, neg)
    want = rl_triton.compute_gae((-x).t().contiguous(), (-x).t().contiguous(), (-x).t().contiguous())
    assert torch.equal(got, want)
    r, v = x.t(), torch.randn(64, 48, device=device).t()
    te = (torch.rand(64, 48, device=device) < 0.1).float().t()
    eager = rl_triton.compute_gae_normalized(r, v, te)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = rl_triton.compute_gae_normalized(r, v, te)
    for _ in range(3):
        for o in out:
            o.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        for o, e in zip(out, eager):
            assert torch.equal(o, e)


def test_time_major_order_of_streams(device, no_flags):
    """Launched on the caller's stream: inputs written there just before are seen."""
    import rl_triton
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        x = torch.zeros(128, 256, device=device)
        for i in range(4):
            x.fill_(float(i))
            got = rl_triton.compute_episodic_prefix_sum(x.t(), torch.zeros_like(x).t())
            assert torch.equal(got[:, -1], torch.full((256,), 128.0 * i, device=device))


@pytest.mark.parametrize("op,boot,shape,copied", [
    ("prefix_sum", "none", (16, 512), False), ("prefix_sum", "none", (16, 1024), True),
    ("prefix_sum", "none", (600, 2048), False), ("gae", "full", (16, 1024), False), ("gae", "full", (16, 2048), True),
    ("vtrace", "row", (64, 2048), True), ("retrace", "none", (16, 1024), False), ("retrace", "none", (16, 2048), True),
    ("gae_normalized_masked", "row", (64, 2048), True), ("discounted_returns", "none", (64, 2048), True)],
    ids=lambda v: f"{v[0]}x{v[1]}" if isinstance(v, tuple) else None)
def test_captured_calls_take_the_faster_form(op, boot, shape, copied, device, no_flags):
    """In a graph the device's time is all that counts: calls of few environments and many steps are
    captured as copies and the row kernel (the bits of the call on contiguous arrays), others as the
    time-major kernel (the bits of the eager call).  Eager calls take the kernel."""
    from rl_triton import _native
    inp, params = _inputs(op, shape, boot, 0.02 if boot == "full" else 0.0)
    d = _columns(inp, device)
    rows = {k: None if v is None else v.contiguous() for k, v in d.items()}
    before = _native.fast.launched()
    want = [t.clone() for t in _call(op, d, params)]
    assert _native.fast.launched() == before + 1
    if copied:
        # two launches of a normalised call have the bits of its one launch
        want = [t.clone() for t in _call(op, rows, params)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    before = _native.fast.launched()
    with torch.cuda.graph(graph):
        got = _call(op, d, params)
    assert _native.fast.launched() - before == (0 if copied else 1)
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert torch.equal(g, w)
    del graph
