"""The recurrences of groups of several XCDs (cut along the contraction and the columns, on the bf16 matrix cores): the edges of
their geometry against the fp64 oracle, and values whose parts would overflow or are not finite."""
import numpy as np
import pytest

from test_gpu_split_recurrence import BOUND, backward, backward_reference, forward, reference
from util import dev, host, problem, relerr

pytestmark = pytest.mark.gpu

# Groups of two XCDs (up to 768 and 1 024 units), four (1 280) and all eight (1 536, 2 048), each with the fewest and most units
# that it takes, a unit beyond whole quads, rows that do not start on 16 bytes; one batch tile per group, two and more, full
# and with a single row.
SHAPES = [(4, 49, 641), (5, 64, 768), (4, 97, 737), (4, 113, 766), (4, 64, 833), (6, 50, 1000), (4, 128, 1024), (5, 33, 1021),
          (4, 1, 1219), (7, 16, 1280), (5, 49, 1277), (4, 100, 1268), (9, 3, 1284), (4, 18, 1536), (6, 49, 1535), (4, 1, 1540),
          (5, 64, 2048), (4, 35, 2045), (4, 130, 1537)]


@pytest.mark.parametrize("T,N,H", SHAPES)
@pytest.mark.parametrize("training,zoneout", [(True, 0.2), (False, 0.2), (True, 0.0)])
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_forward(cell, training, zoneout, T, N, H):
    print("cut recurrence", cell, training, zoneout, T, N, H, flush=True)
    p = problem(T + N + H, T, N, 18, H, 4 if cell == "lstm" else 3, zoneout)
    for ours, theirs in zip(forward(cell, p, training, zoneout), reference(cell, p, training, zoneout)):
        assert relerr(host(ours), theirs) < BOUND


@pytest.mark.parametrize("T,N,H", SHAPES)
@pytest.mark.parametrize("zoneout", [0.0, 0.2])
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_backward(cell, zoneout, T, N, H):
    print("cut backward recurrence", cell, zoneout, T, N, H, flush=True)
    p = problem(T + N + H, T, N, 12, H, 4 if cell == "lstm" else 3, zoneout)
    states = reference(cell, p, True, zoneout)
    # (the same bound as for the split recurrences: the exchange's last bit, T * N terms of the weights' gradients)
    ours, theirs = backward(cell, p, states), backward_reference(cell, p, states)
    for name in ours:
        assert relerr(ours[name], theirs[name]) < 2.0 ** -18, name


EXTREME = [(4, 50, 700), (4, 20, 1290), (5, 70, 1540)]
MANY_NANS = (6, 40, 1300)


@pytest.mark.parametrize("what", ["state", "state_inf", "weight", "weight_inf", "nan"])
@pytest.mark.parametrize("T,N,H", EXTREME)
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_values_that_do_not_split(cell, T, N, H, what):
    """Where fp32 arithmetic gives a finite value it is that value; elsewhere neither is finite."""
    print("cut recurrence, extreme values", cell, T, N, H, what, flush=True)
    p = problem(5 + N, T, N, 13, H, 4 if cell == "lstm" else 3)
    p["h0"][3, 7], p["R"][9, 11] = {"state": (2.0 ** 110, 0.01), "state_inf": (np.inf, 0.01), "weight": (0.5, 2.0 ** 110),
                                    "weight_inf": (0.5, -np.inf), "nan": (np.nan, 0.01)}[what]
    p["h0"][:, 9] = 0.5  # no 0 * inf
    with np.errstate(all="ignore"):
        expected = reference(cell, p, False, 0.0)
    for ours, theirs in zip(forward(cell, p, False, 0.0), expected):
        ours = host(ours)
        same = np.isfinite(theirs)
        assert np.array_equal(np.isfinite(ours), same)
        assert np.array_equal(np.isnan(ours), np.isnan(theirs))
        large = np.abs(theirs) > 2.0 ** 40  # the state itself, where a cell keeps some of it
        ordinary = same & ~large
        assert np.max(np.abs(ours[ordinary] - theirs[ordinary])) < BOUND * max(1.0, np.max(np.abs(theirs[ordinary])))
        if np.any(same & large):
            assert np.max(np.abs(ours[same & large] / theirs[same & large] - 1.0)) < 1e-5


@pytest.mark.parametrize("what", ["gradient", "gradient_large", "gradient_inf", "weight", "weight_inf", "nan"])
@pytest.mark.parametrize("T,N,H", EXTREME)
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_backward_values_that_do_not_split(cell, T, N, H, what):
    """Every gradient is finite, infinite and not a number where the reference is; those that are no sums over the rows are equal
    where finite, batch row 5, which has the extreme gradient, by itself."""
    print("cut backward recurrence, extreme values", cell, T, N, H, what, flush=True)
    p = problem(9 + N, T, N, 8, H, 4 if cell == "lstm" else 3)
    states = reference(cell, p, True, 0.0)
    p["dh_new"][3, 5, 6], p["R"][9, 11] = {"gradient": (2.0 ** 60, 0.01), "gradient_large": (2.0 ** 108, 0.01),
                                           "gradient_inf": (np.inf, 0.01), "weight": (1.0, 2.0 ** 40),
                                           "weight_inf": (1.0, np.inf), "nan": (np.nan, 0.01)}[what]
    with np.errstate(all="ignore"):
        ours, theirs = backward(cell, p, states), backward_reference(cell, p, states)
    for name in theirs:
        a, b = ours[name], theirs[name]
        assert np.array_equal(np.isnan(a), np.isnan(b)), name
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), name
        if name in ("dh0", "dc0", "dx", "dv"):
            row = np.broadcast_to((np.arange(N) == 5)[:, None], b.shape)
            for part in (np.isfinite(b) & row, np.isfinite(b) & ~row):
                if np.any(part):
                    assert np.max(np.abs(a[part] - b[part])) <= 1e-5 * np.max(np.abs(b[part])), name


def test_states_that_are_no_numbers():
    """A layer that has diverged: every state is a NaN, and so is every result, with no sum formed again for it."""
    import time
    import torch
    T, N, H = MANY_NANS
    print("cut recurrence, NaNs", T, N, H, flush=True)
    p = problem(3, T, N, 16, H, 4)
    p["h0"][:] = np.nan
    forward("lstm", p, True, 0.0)
    torch.cuda.synchronize()
    start = time.perf_counter()
    h, c, v = forward("lstm", p, True, 0.0)
    assert torch.isnan(h[1:]).all() and torch.isnan(v).all()
    assert time.perf_counter() - start < 1.0


@pytest.mark.parametrize("N,H", [(50, 700), (20, 1300)])
@pytest.mark.parametrize("cell,training", [("lstm", False), ("lstm", True), ("gru", False), ("gru", True)])
def test_dropconnect_and_run_to_run(cell, training, N, H):
    """The masked weights give what R masked beforehand gives, and a pass what it gave before, bit for bit, also where the
    lent memory is what is stated for the sizes."""
    import torch
    from haste_amd import ops
    T, C = 5, 15
    zoneout = 0.2 if training else 0.0
    p = problem(77 + N, T, N, C, H, 4 if cell == "lstm" else 3, zoneout)
    keep = (np.random.default_rng(N).uniform(size=p["R"].shape) >= 0.3).astype(np.float64)
    scale = 2.0
    mask = dev(p["mask"]) if zoneout else torch.empty(0, device="cuda")
    x, h0, c0, W, b, b2 = (dev(p[k]) for k in ("x", "h0", "c0", "W", "b", "b2"))

    def run(R, *dropconnect):
        if cell == "lstm":
            return ops.lstm_forward(training, zoneout, x, h0, c0, W, R, b, mask, *dropconnect)
        out = ops.gru_forward(training, zoneout, x, h0, W, R, b, b2, mask, *dropconnect)
        return out if training else out[:1]  # (the second one is written in training only)

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        masked = (dev(p["R"]), dev(keep), scale)
        want = run(dev(p["R"] * keep * scale))
        first, again = run(*masked), run(*masked)
        lent = torch.empty(ops.workspace_bytes(T, N, C, H), dtype=torch.uint8, device="cuda")
        try:
            ops.set_workspace(lent)
            in_lent = run(*masked)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                captured = run(*masked)
            replays = []
            for _ in range(3):
                for t in captured:
                    t.zero_()
                graph.replay()
                replays.append([t.clone() for t in captured])
            stream.synchronize()
            ops.stream_status()
        finally:
            ops.set_workspace(None)
    states = 2 if cell == "lstm" else 1  # (the LSTM's third one is scratch where it does not train)
    for got in [first, again, in_lent] + replays:
        assert all(torch.equal(a, b) for a, b in zip(got[:None if training else states], want))


def test_graph_replay():
    """Captured with a lent workspace and replayed: what the eager pass gives, each time."""
    import torch
    from haste_amd import ops
    T, N, C, H = 4, 40, 16, 1300
    p = problem(11, T, N, C, H, 4)
    args = [dev(p[k]) for k in ("x", "h0", "c0", "W", "R", "b")]
    none = torch.empty(0, device="cuda")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        expected = ops.lstm_forward(True, 0.0, *args, none)
        lent = torch.empty(ops.workspace_bytes(T, N, C, H), dtype=torch.uint8, device="cuda")
        ops.set_workspace(lent)
        ops.lstm_forward(True, 0.0, *args, none)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = ops.lstm_forward(True, 0.0, *args, none)
        for _ in range(3):
            for t in out:
                t.zero_()
            graph.replay()
            eager = ops.lstm_forward(True, 0.0, *args, none)
            stream.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, expected))
            assert all(torch.equal(a, b) for a, b in zip(eager, expected))
        ops.set_workspace(None)
