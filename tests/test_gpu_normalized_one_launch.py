"""compute_gae_normalized in one launch (finish_normalized in csrc/rlk_engine.hpp): the bits of the
two-launch form, also when workgroups stop waiting and leave raw advantages for others to
normalise."""
import pytest
import torch

from _common import make_inputs, to_device

pytestmark = pytest.mark.gpu

# one workgroup, several with a partial last one, one row per workgroup (strided, whole rows), as
# many workgroups as fit at once and more (two launches), rows split into tiles (two launches)
SHAPES = [(2, 3), (5, 1), (4, 128), (300, 33), (33, 257), (600, 500), (16, 2048), (300, 1100), (3, 5000),
          (512, 6000), (200, 9000), (4096, 128), (16384, 128), (20000, 128), (3, 40000)]


def _call(d, params, columns=False):
    import rl_triton
    if columns:
        d = {k: v if v is None or v.dim() < 2 else v.t().contiguous().t() for k, v in d.items()}
    return rl_triton.compute_gae_normalized(d["rewards"], d["values"], d["terminateds"], d.get("truncateds"),
                                            bootstrap_values=d.get("bootstrap_values"),
                                            last_value=d.get("last_value"), mask=d.get("mask"), **params)


def _two_launches(d, params, columns=False):
    """The same call captured: graph replays would repeat the one-launch form's call count."""
    _call(d, params, columns)
    torch.cuda.synchronize()
    if columns:
        d = {k: v if v is None or v.dim() < 2 else v.t().contiguous().t() for k, v in d.items()}
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = _call(d, params)
    g.replay()
    torch.cuda.synchronize()
    return [t.clone() for t in out]


@pytest.fixture(params=[None, 0, 1], ids=["waiting", "not_waiting", "one_more_read"])
def polls(request, monkeypatch):
    """How often a workgroup looks again for the others' statistics: as shipped, never, once."""
    from rl_triton import _native
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    lib = _native.load()
    if request.param is not None:
        lib.rlk_debug_lookback(-1, request.param)
    yield request.param
    lib.rlk_debug_lookback(-1, -1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_bits_of_two_launches(shape, masked, dtype, polls, device):
    op = "gae_normalized_masked" if masked else "gae_normalized"
    inp, params = make_inputs(op, *shape, seed=sum(shape), p_trunc=0.02, boot="full")
    d = to_device(inp, device, dtype)
    want = _two_launches(d, params)
    for _ in range(5):
        for g, w in zip(_call(d, params), want):
            assert torch.equal(g.view(torch.int16), w.view(torch.int16)), f"{op}{shape} {dtype}"


@pytest.mark.parametrize("shape", [(5, 3), (100, 33), (300, 100), (4100, 128), (70, 256), (64, 300)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_bits_of_two_launches_time_major(shape, polls, device):
    inp, params = make_inputs("gae_normalized", *shape, seed=7, boot="row")
    d = to_device(inp, device)
    want = _two_launches(d, params, columns=True)
    for _ in range(5):
        for g, w in zip(_call(d, params, columns=True), want):
            assert torch.equal(g, w), f"{shape}"


def test_streams_and_call_limit(device, monkeypatch):
    """Calls on two streams at once keep their own buffers; a buffer is zeroed again at the call
    limit."""
    from rl_triton import _native
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    inp, params = make_inputs("gae_normalized", 1024, 128, seed=3, boot="row")
    d = to_device(inp, device)
    want = _two_launches(d, params)
    prev = _native.fast.set_workspace_max_calls(3)
    clears = _native.fast.sync_clears()
    try:
        streams = [torch.cuda.Stream() for _ in range(2)]
        torch.cuda.synchronize()
        outs = []
        for i in range(10):
            for s in streams:
                with torch.cuda.stream(s):
                    outs.append(_call(d, params))
        torch.cuda.synchronize()
        # ten calls on each stream, at most three between two clears
        assert _native.fast.sync_clears() - clears >= 2 * 3
        for out in outs:
            for g, w in zip(out, want):
                assert torch.equal(g, w)
    finally:
        _native.fast.set_workspace_max_calls(prev)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("trunc", [False, True])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", [(200, 9000), (130, 9217)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_four_segment_rows(shape, masked, trunc, dtype, polls, device):
    """Four segments per thread, with and without truncations (instances of their own): a workgroup
    that stops waiting marks its raw advantages only once they are written."""
    op = "gae_normalized_masked" if masked else "gae_normalized"
    inp, params = make_inputs(op, *shape, seed=sum(shape), p_trunc=0.02 if trunc else 0.0, boot="full" if trunc else "row")
    d = to_device(inp, device, dtype)
    want = _two_launches(d, params)
    for _ in range(5):
        for g, w in zip(_call(d, params), want):
            assert torch.equal(g.view(torch.int16), w.view(torch.int16)), f"{op}{shape} {dtype}"


def _marks():
    """How many workgroups of the last one-launch call on each stream stopped waiting: words of the
    buffer's state part (behind 8 words and 4 per workgroup, 512 workgroups) with that call's epoch,
    marked raw (1) or raw and normalised by another workgroup (2)."""
    from rl_triton import _native
    raw = claimed = 0
    for _, epoch, buf in _native.fast.norm_syncs():
        state = buf.view(torch.int64)[8 + 4 * 512:].cpu()
        assert state.numel() == 512
        mine = state[(state >> 48) & 0xffff == epoch] & 0xffff
        raw, claimed = raw + int((mine == 1).sum()), claimed + int((mine == 2).sum())
    return raw, claimed


def _one_launches():
    from rl_triton import _native
    return _native.fast.one_launches()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", [(64, 64), (1024, 128), (256, 2048), (300, 1100), (512, 2052), (512, 6000), (257, 6148),
                                   (300, 6656), (300, 6660), (300, 7000), (512, 7168), (257, 7172), (300, 8192),
                                   (256, 9000), (400, 9000), (300, 12000), (256, 16384)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_no_workgroup_stops_waiting(shape, masked, dtype, device, monkeypatch):
    """A call takes one launch only where its workgroups are resident together: with nothing else on
    the GPU none of them runs out of polls.  (Twelve waves of four segments per thread and more are
    where a CU's register count and its SIMDs' wave slots differ.)"""
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    op = "gae_normalized_masked" if masked else "gae_normalized"
    inp, params = make_inputs(op, *shape, seed=1, boot="row")
    d = to_device(inp, device, dtype)
    for _ in range(3):
        torch.cuda.synchronize()
        _call(d, params)
        torch.cuda.synchronize()
        assert _marks() == (0, 0)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", [(1024, 128), (256, 4096), (200, 9000), (130, 9217)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_raw_advantages_are_claimed_once(shape, masked, device, monkeypatch):
    """Workgroups that never look again stop waiting, unless all others came first: each one marked
    raw is taken by one that has all statistics, and none is left."""
    from rl_triton import _native
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    op = "gae_normalized_masked" if masked else "gae_normalized"
    inp, params = make_inputs(op, *shape, seed=2, boot="row")
    d = to_device(inp, device)
    want = _two_launches(d, params)
    _native.load().rlk_debug_lookback(-1, 0)
    try:
        claimed = 0
        for _ in range(5):
            before = _one_launches()
            got = _call(d, params)
            torch.cuda.synchronize()
            assert _one_launches() == before + 1
            raw, c = _marks()
            claimed += c
            assert raw == 0
            for g, w in zip(got, want):
                assert torch.equal(g, w)
        assert claimed > 0
    finally:
        _native.load().rlk_debug_lookback(-1, -1)


# (shape, one launch unmasked, one launch masked): both sides of each line of one_launch_blocks
@pytest.mark.parametrize("shape,plain,masked", [
    ((64, 64), True, True), ((4096, 128), True, True), ((4097, 128), False, False), ((256, 1024), True, True),
    ((1024, 1000), False, False), ((384, 1028), True, True), ((385, 1028), True, False), ((512, 2048), True, False),
    ((513, 2048), False, False), ((256, 2047), True, True), ((257, 2047), False, False), ((512, 2049), True, True),
    ((513, 2049), False, False), ((512, 6000), True, True), ((300, 7000), True, False), ((512, 8192), True, False),
    ((256, 9000), True, True), ((257, 9000), True, False), ((3, 16385), False, False)],
    ids=lambda s: f"{s[0]}x{s[1]}" if isinstance(s, tuple) else None)
def test_which_calls_take_one_launch(shape, plain, masked, device, monkeypatch):
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    for op, want in (("gae_normalized", plain), ("gae_normalized_masked", masked)):
        inp, params = make_inputs(op, *shape, seed=4, boot="row")
        d = to_device(inp, device)
        before = _one_launches()
        _call(d, params)
        assert _one_launches() - before == want, op
        before = _one_launches()
        _two_launches(d, params)
        assert _one_launches() - before == want, f"{op}: a captured call"


@pytest.mark.parametrize("shape,want", [((64, 64), True), ((4096, 128), True), ((4112, 128), False), ((100, 256), True),
                                        ((100, 257), False)], ids=lambda s: f"{s[0]}x{s[1]}" if isinstance(s, tuple) else None)
def test_which_time_major_calls_take_one_launch(shape, want, device, monkeypatch):
    monkeypatch.delenv("RL_TRITON_CORRECTNESS_WARNINGS", raising=False)
    inp, params = make_inputs("gae_normalized", *shape, seed=5, boot="row")
    before = _one_launches()
    _call(to_device(inp, device), params, columns=True)
    assert _one_launches() - before == want
